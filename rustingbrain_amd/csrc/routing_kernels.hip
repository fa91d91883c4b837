// Router, dispatch and combine kernels of the mixture-of-experts forward pass
// for gfx950 (wave64).
//
//   logits_kernel   router logits in the reference's eight-lane `dot` order
//   router_kernel   softmax, log-sum-exp, deterministic top-k, per-block ranks
//                   and histogram, per-block partial sums for the auxiliary losses
//   route_rows_kernel, route_fused_kernel   both in one launch, by calls of up to 256 K pairs (plan_router)
//   dispatch_kernel prefix scan over blocks and experts, stable permutation
//                   (slot -> position), optional row gather; block 0 also writes
//                   the tile table of the grouped products and the two losses
//   combine_kernel  gate-weighted sum in ascending expert order, then the
//                   shared expert, then the optional residual
//
// Nothing here uses floating-point atomics: every sum has a fixed order, so two
// runs give the same bits.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <type_traits>

#include "layout_device.h"
#include "routing_device.h"

namespace rbmoe {

size_t router_lds_bytes(int E, int k) {
    return router_fixed_bytes(E, k);
}

// ---------------------------------------------------------------------------
// logits_kernel: logits[t, e] = dot(x[t, :], w[e, :]) (+ bias[e]) in the order of the
// reference's eight-lane `dot` (src/matrix.rs:26-40): lanes[c % 8] += x[c] * w[c] in
// increasing c (a rounded multiply, then a rounded add), a scalar `rest` for the columns
// past the last multiple of 8, lanes folded left to right, rest added last.
//
// A workgroup owns 64 tokens x 8 experts: 8 waves, lane = token, one expert per wave, so a
// router row is wave-uniform and is fetched with scalar loads (it costs neither vector
// memory bandwidth nor LDS), 64 columns at a time so that their latency is paid once per
// batch.  The token rows are staged through LDS in slices of kLogitChunk columns (16-byte
// pieces, rows padded by one piece so that a wave's 64 row reads spread over all banks).
// ---------------------------------------------------------------------------
constexpr int kLogitTokens = 64;
constexpr int kLogitChunk = 256;
constexpr int kLogitBatch = 8;  // pieces (of 8 columns) per batch of scalar loads

template <typename XT>
struct XPiece;  // 8 consecutive elements of a token row
template <>
struct XPiece<bf16_t> {
    typedef uint4 raw_t;
    static __device__ __forceinline__ void widen(const raw_t& a, float (&v)[8]) {
        v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
        v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
        v[4] = __uint_as_float(a.z << 16); v[5] = __uint_as_float(a.z & 0xffff0000u);
        v[6] = __uint_as_float(a.w << 16); v[7] = __uint_as_float(a.w & 0xffff0000u);
    }
};
template <>
struct XPiece<float> {
    struct raw_t {
        float4 a, b;
    };
    static __device__ __forceinline__ void widen(const raw_t& r, float (&v)[8]) {
        v[0] = r.a.x; v[1] = r.a.y; v[2] = r.a.z; v[3] = r.a.w;
        v[4] = r.b.x; v[5] = r.b.y; v[6] = r.b.z; v[7] = r.b.w;
    }
};

// NE = experts (= waves) per workgroup.
// (bf16 without AHEAD: 6 waves per SIMD, i.e. three workgroups on a compute unit, is what the launches of many
// workgroups are tuned for - the bound keeps a later edit from quietly costing one of them)
// `rows16` (f32 rows only, or null): a bf16 copy of the rows, rounded to nearest even, for the expert products of a
// layer whose weights are bf16 or int8 - written on the way by the workgroups of the first group of experts, which
// have every piece of their rows in hand anyway (widths that are multiples of 8).
// WIDE (bf16 rows): the rows are widened to f32 once, on their way into LDS, instead of by each of the NE waves
// that read them (one of the three vector instructions per element); a slice is then half as many columns, so
// that a workgroup takes no more LDS and as many of them fit a compute unit.  So it is for f32 rows in launches of many
// workgroups: four on a compute unit instead of two (64 experts of 704, d 1024, 16384 f32 rows 823.7 -> 803 us a forward, while
// those were routed here).
// NL = 32: the logits of a quantized router, in the order of dot_lanes::<32> (src/quantized.rs:154-177): lanes[c % 32] +=
// x[c] * f32(q[c]), the scalar rest from the last multiple of 32 on, and the whole times the row's `scale` (:61).  `wr` then
// holds the int8 weights widened once, at their upload: a whole number in f32 is fetched like any other router weight.
// For bf16 rows; bound by the vector units like the other order.  us a forward with a thread a product over the int8 rows
// (logits_q8_kernel: 64 lines of them a load) / with this: 64 experts of 704, d 1024, 16384 tokens 734.6 / 639.7, 4096
// 209.0 / 202.3; 16 experts of 256, d 1024, 16384 tokens 171.9 / 140.4; 32 of 256, 5000 tokens 107.1 / 85.5; 8 of 256, d 768,
// 12000 tokens 107.1 / 95.1; 128 of 64, d 512, one token 55.7 / 51.6, 64 tokens 61.1 / 58.0.
template <typename XT, int NE, bool AHEAD, bool WIDE = false, int NL = 8>
__global__ __launch_bounds__(NE * 64, (!AHEAD && sizeof(XT) == 2) ? 6 : 2) void logits_kernel(const XT* __restrict__ x,
                                                                const float* __restrict__ wr,
                                                                const float* __restrict__ bias, int T, int d, int E,
                                                                float* __restrict__ logits,
                                                                bf16_t* __restrict__ rows16,
                                                                const float* __restrict__ scale) {
    static_assert(!WIDE || sizeof(XT) == 2, "only bf16 rows are widened");
    static_assert(NL == 8 || (NL == 32 && sizeof(XT) == 2), "32 lanes: bf16 rows");
    typedef typename XPiece<XT>::raw_t piece_t;
    typedef typename std::conditional<WIDE, float, XT>::type ST;  // the element type of the staged rows
    typedef typename XPiece<ST>::raw_t spiece_t;
    constexpr int kChunk = !AHEAD && sizeof(ST) == 4 ? kLogitChunk / 2 : kLogitChunk;
    constexpr int PIECES = kChunk / 8;  // pieces per row per slice
    constexpr int ROWB = PIECES * (int)sizeof(spiece_t) + 16;  // bytes of a staged row: 16 of padding, so that the lanes' rows start in different banks
    __shared__ __align__(16) unsigned char xs_raw[kLogitTokens * ROWB];
    auto staged = [&](int r, int q) -> spiece_t* {
        return reinterpret_cast<spiece_t*>(xs_raw + (size_t)r * ROWB + (size_t)q * sizeof(spiece_t));
    };
    auto put = [&](int r, int q, const piece_t& v) {
        if constexpr (WIDE) {
            float f[8];
            XPiece<XT>::widen(v, f);
            spiece_t o;
            o.a = make_float4(f[0], f[1], f[2], f[3]);
            o.b = make_float4(f[4], f[5], f[6], f[7]);
            *staged(r, q) = o;
        } else {
            *staged(r, q) = v;
        }
    };
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t0 = blockIdx.x * kLogitTokens;
    const int nt = min(kLogitTokens, T - t0);
    constexpr int kLogitThreads = NE * 64;
    const int e = blockIdx.y * NE + wave;  // this wave's expert
    const bool has = e < E;
    const float* w0 = wr + (size_t)(has ? e : 0) * d;
    const int tail = d - d % NL;
    float la[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) la[l] = 0.0f;
    const bool vec = d % 8 == 0 && (NL == 8 || (reinterpret_cast<uintptr_t>(x) & 15) == 0);
    constexpr int TURN = NL / 8;                                // pieces of one turn of the column lanes
    constexpr int BATCH = NL == 8 ? kLogitBatch : TURN;         // (32 sums leave registers for half a batch)
    static_assert(PIECES % BATCH == 0 && BATCH % TURN == 0, "a slice is whole turns");
    // A slice's pieces travel global -> registers -> LDS.  AHEAD: the loads of the next slice are issued
    // before the products of the current one, so their latency is covered by arithmetic - for launches of few
    // workgroups; with several workgroups on a compute unit they cover for each other, and the registers the
    // pieces in flight occupy would cost one of them.
    constexpr int MAXP = (kLogitTokens * PIECES + kLogitThreads - 1) / kLogitThreads;
    piece_t pre[MAXP];
    const bool copy16 = sizeof(XT) == 4 && rows16 != nullptr && blockIdx.y == 0;
    auto load_piece = [&](int r, int c) {  // eight elements of row r from column c (zeros past the last row)
        piece_t v = {};
        if (r < nt) {
            const XT* src = x + (size_t)(t0 + r) * d + c;
            if (vec) {
                v = *reinterpret_cast<const piece_t*>(src);
                if constexpr (sizeof(XT) == 4) {
                    if (copy16) {
                        float f[8];
                        XPiece<XT>::widen(v, f);
                        uint4 o;
                        o.x = f32_to_bf16_bits(f[0]) | ((uint32_t)f32_to_bf16_bits(f[1]) << 16);
                        o.y = f32_to_bf16_bits(f[2]) | ((uint32_t)f32_to_bf16_bits(f[3]) << 16);
                        o.z = f32_to_bf16_bits(f[4]) | ((uint32_t)f32_to_bf16_bits(f[5]) << 16);
                        o.w = f32_to_bf16_bits(f[6]) | ((uint32_t)f32_to_bf16_bits(f[7]) << 16);
                        *reinterpret_cast<uint4*>(rows16 + (size_t)(t0 + r) * d + c) = o;
                    }
                }
            } else {  // rows are not 16-byte aligned: gather the eight elements
                XT tmp[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) tmp[j] = src[j];
                v = *reinterpret_cast<const piece_t*>(tmp);
            }
        }
        return v;
    };
    auto fetch = [&](int c0) {
        const int np = min(PIECES, (tail - c0) / 8);
#pragma unroll
        for (int u = 0; u < MAXP; ++u) {
            const int idx = tid + u * kLogitThreads;  // over the full 64 x PIECES grid: no division by np
            const int r = idx / PIECES, q = idx % PIECES;
            pre[u] = (r < kLogitTokens && q < np) ? load_piece(r, c0 + 8 * q) : piece_t{};
        }
    };
    if (AHEAD && tail > 0) fetch(0);
    for (int c0 = 0; c0 < tail; c0 += kChunk) {
        const int np = min(PIECES, (tail - c0) / 8);  // pieces in this slice
        __syncthreads();
        if (AHEAD) {
#pragma unroll
            for (int u = 0; u < MAXP; ++u) {
                const int idx = tid + u * kLogitThreads;
                const int r = idx / PIECES, q = idx % PIECES;
                if (r < kLogitTokens && q < np) put(r, q, pre[u]);
            }
        } else {
            for (int idx = tid; idx < kLogitTokens * np; idx += kLogitThreads) {
                const int r = idx / np, q = idx - r * np;
                put(r, q, load_piece(r, c0 + 8 * q));
            }
        }
        __syncthreads();
        if (AHEAD && c0 + kChunk < tail) fetch(c0 + kChunk);
        if (has) {
            const float* wa = w0 + c0;
            int q = 0;
            for (; q + BATCH <= np; q += BATCH) {
                // one batch: its router weights into scalar registers, its token pieces from LDS
                float wv[8 * BATCH];
#pragma unroll
                for (int j = 0; j < 8 * BATCH; ++j) wv[j] = wa[8 * q + j];
                spiece_t xp[BATCH];
#pragma unroll
                for (int b = 0; b < BATCH; ++b) xp[b] = *staged(lane, q + b);
#pragma unroll
                for (int b = 0; b < BATCH; ++b) {
                    float xv[8];
                    XPiece<ST>::widen(xp[b], xv);
#pragma unroll
                    for (int l = 0; l < 8; ++l) {
                        float& sum = la[8 * (b % TURN) + l];
                        sum = __fadd_rn(sum, __fmul_rn(xv[l], wv[8 * b + l]));
                    }
                }
            }
            if constexpr (BATCH > TURN)
                for (; q < np; ++q) {
                    static_assert(TURN == 1, "one piece a turn");
                    float xv[8];
                    XPiece<ST>::widen(*staged(lane, q), xv);
#pragma unroll
                    for (int l = 0; l < 8; ++l) la[l] = __fadd_rn(la[l], __fmul_rn(xv[l], wa[8 * q + l]));
                }
        }
    }
    if (lane < nt && has) {
        const XT* xr = x + (size_t)(t0 + lane) * d;
        float rest = 0.0f;
        for (int c = tail; c < d; ++c) rest = __fadd_rn(rest, __fmul_rn(to_f32(xr[c]), w0[c]));
        float sum = 0.0f;
#pragma unroll
        for (int l = 0; l < NL; ++l) sum = __fadd_rn(sum, la[l]);
        float v = __fadd_rn(sum, rest);
        if constexpr (NL == 32) v = __fmul_rn(v, scale[e]);
        if (bias) v = __fadd_rn(v, bias[e]);
        logits[(size_t)(t0 + lane) * E + e] = v;
    }
}

// ---------------------------------------------------------------------------
// logits_q8_kernel: the logits of a quantized router, one thread per (token, expert).  The reference's order
// (dot_lanes::<32>, src/quantized.rs:154-177, taken on machines with AVX2, :179-196): lanes[c % 32] += x[c] * f32(q[c])
// over the whole chunks of 32 columns, a scalar rest over the tail, the lanes folded from 0.0 in lane order, plus the
// rest, times the row's scale (:61); every product and every sum rounded by itself.  Any width.  For f32 rows: there
// logits_kernel's own order of lanes is no faster in large launches (us a forward, this / logits_kernel<NL = 32>: 12000
// tokens, d 768, 8 experts 115.6 / 120.8; 5000, d 1024, 32 experts 113.5 / 135.5; 3000, d 512, 64 experts 69.6 / 79.9; 8192,
// d 768, 16 experts 169.9 / 163.0); bf16 rows are routed there.
// ---------------------------------------------------------------------------
template <typename XT>
__global__ __launch_bounds__(256) void logits_q8_kernel(const XT* __restrict__ x, const int8_t* __restrict__ q,
                                                        const float* __restrict__ scale, const float* __restrict__ bias,
                                                        int T, int d, int E, float* __restrict__ P) {
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long long)T * E) return;
    const int t = (int)(idx / E), e = (int)(idx - (long long)t * E);
    const XT* const xr = x + (size_t)t * d;
    const int8_t* const qr = q + (size_t)e * d;
    float lanes[32];
#pragma unroll
    for (int l = 0; l < 32; ++l) lanes[l] = 0.0f;
    const int tail = d - d % 32;
    for (int c = 0; c < tail; c += 32) {
#pragma unroll
        for (int l = 0; l < 32; ++l)
            lanes[l] = __fadd_rn(lanes[l], __fmul_rn(to_f32(xr[c + l]), (float)qr[c + l]));
    }
    float rest = 0.0f;
    for (int c = tail; c < d; ++c) rest = __fadd_rn(rest, __fmul_rn(to_f32(xr[c]), (float)qr[c]));
    float sum = 0.0f;
#pragma unroll
    for (int l = 0; l < 32; ++l) sum = __fadd_rn(sum, lanes[l]);
    float v = __fmul_rn(__fadd_rn(sum, rest), scale[e]);
    if (bias) v = __fadd_rn(v, bias[e]);
    P[idx] = v;
}

// ---------------------------------------------------------------------------
// route_fused_kernel: the logits AND everything behind them for the 32 tokens of a router block, in one workgroup
// - one launch and one trip of the logits through memory less than logits_kernel + router_kernel.  A workgroup
// must then hold every expert of its tokens, and with 32 tokens a wave's 64 lanes are two experts side by side:
// lane = (token, half), wave w takes the experts 2 w + half (+ 16, + 32, ... for more than 16 experts).  The router
// rows are no longer uniform over a wave, so they are staged in LDS beside the token rows, a slice of columns at a
// time, and read from there (one address per half-wave: a broadcast).  The arithmetic is logits_kernel's, element by
// element: lanes[c % 8] += x[c] * w[c] in increasing c, a rounded multiply and a rounded add, the lanes folded left
// to right (widths that are multiples of 8: no tail).
// Dynamic LDS: the arrays of router_tail, then 32 token rows and E router rows of one slice.
// NI = experts per lane = ceil(E / 16).
// ---------------------------------------------------------------------------
__host__ __device__ static size_t fused_lds_bytes(int E, int k, int cols, size_t xsize) {
    return router_fixed_bytes(E, k) + (size_t)kRouterTokens * (cols * xsize + 16) + (size_t)E * (cols * 4 + 16);
}

// WIDE (bf16 rows): the token rows are widened to f32 once, on their way into LDS, instead of by each of the 16
// lanes that read an element (a shift or a mask per element and lane: a fifth of the kernel's vector
// instructions); the staged slice then takes twice the LDS, so the launcher asks for it only where that fits.
template <typename XT, int NI, bool WIDE>
__global__ __launch_bounds__(kRouterThreads) void route_fused_kernel(
    const XT* __restrict__ x, const float* __restrict__ wr, const float* __restrict__ bias,
    const uint8_t* __restrict__ valid, int T, int d, int E, int k, int cols, float* __restrict__ P,
    float* __restrict__ lse, int* __restrict__ expert_of, float* __restrict__ gate_of,
    int* __restrict__ rank_in_block, int* __restrict__ blockcnt, float* __restrict__ partial,
    bf16_t* __restrict__ rows16) {
    typedef typename XPiece<XT>::raw_t piece_t;
    typedef typename std::conditional<WIDE, float, XT>::type ST;  // the element type of the staged token rows
    typedef typename XPiece<ST>::raw_t spiece_t;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int TB = kRouterTokens;
    const int ES = E | 1;
    float* const prob = reinterpret_cast<float*>(lds_raw);
    const int xpitch = cols * (int)sizeof(ST) + 16, wpitch = cols * 4 + 16;  // bytes; + 16: rows start in different banks
    unsigned char* const xs = lds_raw + router_fixed_bytes(E, k);
    unsigned char* const ws = xs + (size_t)TB * xpitch;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = lane & 31, half = lane >> 5;
    const int blk = blockIdx.x;
    const int t0 = blk * TB;
    const int nt = min(TB, T - t0);

    float la[NI][8];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int l = 0; l < 8; ++l) la[i][l] = 0.0f;

    // A slice travels global -> registers -> LDS; the loads of the next slice are issued before the products of the
    // current one, so that their latency is covered by arithmetic.  A thread moves up to MAXX pieces of token rows
    // (32 rows x 32 pieces at most) and MAXW 16-byte pieces of router rows (E rows x 64 at most) per slice.
    constexpr int MAXX = (kRouterTokens * 32 + kRouterThreads - 1) / kRouterThreads;
    constexpr int MAXW = (NI * 16 * 64 + kRouterThreads - 1) / kRouterThreads;
    piece_t pre_x[MAXX];
    float4 pre_w[MAXW];
    auto fetch = [&](int c0) {
        const int nc = min(cols, d - c0);
        const int np = nc / 8, nq = nc / 4;
#pragma unroll
        for (int u = 0; u < MAXX; ++u) {
            const int idx = tid + u * kRouterThreads;
            const int r = idx / np, q = idx - r * np;
            pre_x[u] = (idx < TB * np && r < nt) ? *reinterpret_cast<const piece_t*>(x + (size_t)(t0 + r) * d + c0 + 8 * q)
                                                 : piece_t{};
        }
#pragma unroll
        for (int u = 0; u < MAXW; ++u) {
            const int idx = tid + u * kRouterThreads;
            const int e = idx / nq, j = idx - e * nq;
            pre_w[u] = idx < E * nq ? *reinterpret_cast<const float4*>(wr + (size_t)e * d + c0 + 4 * j)
                                    : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    };
    auto stage = [&](int c0) {
        const int nc = min(cols, d - c0);
        const int np = nc / 8, nq = nc / 4;
#pragma unroll
        for (int u = 0; u < MAXX; ++u) {
            const int idx = tid + u * kRouterThreads;
            if (idx < TB * np) {
                const int r = idx / np, q = idx - r * np;
                if constexpr (WIDE && sizeof(XT) == 2) {
                    float f[8];
                    XPiece<XT>::widen(pre_x[u], f);
                    float4* const to = reinterpret_cast<float4*>(xs + (size_t)r * xpitch + (size_t)q * sizeof(spiece_t));
                    to[0] = make_float4(f[0], f[1], f[2], f[3]);
                    to[1] = make_float4(f[4], f[5], f[6], f[7]);
                } else {
                    *reinterpret_cast<piece_t*>(xs + (size_t)r * xpitch + (size_t)q * sizeof(piece_t)) = pre_x[u];
                }
                if constexpr (sizeof(XT) == 4) {
                    if (rows16 != nullptr && r < nt) {  // the bf16 copy of f32 rows for the expert products (see logits_kernel)
                        float f[8];
                        XPiece<XT>::widen(pre_x[u], f);
                        uint4 o;
                        o.x = f32_to_bf16_bits(f[0]) | ((uint32_t)f32_to_bf16_bits(f[1]) << 16);
                        o.y = f32_to_bf16_bits(f[2]) | ((uint32_t)f32_to_bf16_bits(f[3]) << 16);
                        o.z = f32_to_bf16_bits(f[4]) | ((uint32_t)f32_to_bf16_bits(f[5]) << 16);
                        o.w = f32_to_bf16_bits(f[6]) | ((uint32_t)f32_to_bf16_bits(f[7]) << 16);
                        *reinterpret_cast<uint4*>(rows16 + (size_t)(t0 + r) * d + c0 + 8 * q) = o;
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < MAXW; ++u) {
            const int idx = tid + u * kRouterThreads;
            if (idx < E * nq) {
                const int e = idx / nq, j = idx - e * nq;
                *reinterpret_cast<float4*>(ws + (size_t)e * wpitch + 16 * j) = pre_w[u];
            }
        }
    };
    fetch(0);
    for (int c0 = 0; c0 < d; c0 += cols) {
        const int nc = min(cols, d - c0);
        const int np = nc / 8;  // pieces of 8 columns in this slice
        __syncthreads();        // the slice before has been consumed
        stage(c0);
        __syncthreads();
        if (c0 + cols < d) fetch(c0 + cols);
        // The LDS reads of piece q + 1 are issued before the arithmetic of piece q, so that their latency is covered
        // by it (two waves on a SIMD do not cover it by themselves).  An expert index past E is clamped: its sums
        // are computed and dropped, which keeps branches out of the loop.
        const unsigned char* const xrow = xs + (size_t)t * xpitch;
        const unsigned char* wrow[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) wrow[i] = ws + (size_t)min(2 * wave + half + 16 * i, E - 1) * wpitch;
        struct Operands {
            spiece_t x;
            float4 wa[NI], wb[NI];
        };
        auto read = [&](Operands& o, int q) {
            o.x = lds_load_ahead<spiece_t>(xrow + (size_t)q * sizeof(spiece_t));
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                o.wa[i] = lds_load_ahead<float4>(wrow[i] + 32 * q);
                o.wb[i] = lds_load_ahead<float4>(wrow[i] + 32 * q + 16);
            }
            __builtin_amdgcn_sched_barrier(0);  // the reads stay in front of the arithmetic that follows
        };
        auto multiply = [&](const Operands& o) {
            float xv[8];
            XPiece<ST>::widen(o.x, xv);
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                la[i][0] = __fadd_rn(la[i][0], __fmul_rn(xv[0], o.wa[i].x));
                la[i][1] = __fadd_rn(la[i][1], __fmul_rn(xv[1], o.wa[i].y));
                la[i][2] = __fadd_rn(la[i][2], __fmul_rn(xv[2], o.wa[i].z));
                la[i][3] = __fadd_rn(la[i][3], __fmul_rn(xv[3], o.wa[i].w));
                la[i][4] = __fadd_rn(la[i][4], __fmul_rn(xv[4], o.wb[i].x));
                la[i][5] = __fadd_rn(la[i][5], __fmul_rn(xv[5], o.wb[i].y));
                la[i][6] = __fadd_rn(la[i][6], __fmul_rn(xv[6], o.wb[i].z));
                la[i][7] = __fadd_rn(la[i][7], __fmul_rn(xv[7], o.wb[i].w));
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // two sets of operand registers take turns, so that nothing is copied between the trips
        Operands oa, ob;
        read(oa, 0);
        for (int q = 0; q < np; q += 2) {
            read(ob, min(q + 1, np - 1));
            multiply(oa);
            read(oa, min(q + 2, np - 1));
            if (q + 1 < np) multiply(ob);
        }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int e = 2 * wave + half + 16 * i;
        if (e < E && t < nt) {
            float sum = 0.0f;
#pragma unroll
            for (int l = 0; l < 8; ++l) sum = __fadd_rn(sum, la[i][l]);
            float v = __fadd_rn(sum, 0.0f);  // the reference adds its (empty) scalar rest: sum + 0
            if (bias) v = __fadd_rn(v, bias[e]);
            prob[t * ES + e] = v;
        }
    }
    __syncthreads();
    router_tail<1, kRouterTokens>(lds_raw, blk, valid, T, E, k, RouteOut{P, lse, expert_of, gate_of}, rank_in_block, blockcnt, partial,
                                  [&](int i, int e) { return prob[i * ES + e]; });
}

// Norm (optional), logits and everything behind them for TB tokens a workgroup (see route_rows_body).
template <typename XT, int TB, int NL, int TT, int EE, bool NORM>
__global__ __launch_bounds__(kRouterThreads, 2) void route_rows_kernel(RouteRowsArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if (a.slice == 0) {  // uniform over the launch
        route_rows_body<XT, TB, NL, TT, EE, NORM>(a, blockIdx.x, 0, a.E, lds_raw);
        __syncthreads();
    } else {
        const int from = blockIdx.y * a.slice, to = min(a.E, from + a.slice);
        RouteRowsArgs own = a;
        if (blockIdx.y != 0) own.xn_out = own.rows16 = nullptr;  // (the first slice writes the rows)
        route_rows_body<XT, TB, NL, TT, EE, NORM>(own, blockIdx.x, from, to, lds_raw);
        __syncthreads();
        if (!last_slice<TB>(a, from, to, lds_raw)) return;
    }
    const float* const prob = reinterpret_cast<const float*>(lds_raw);
    const int ES = a.E | 1;
    router_tail<1, TB>(lds_raw, blockIdx.x, a.valid, a.T, a.E, a.k, RouteOut{a.P, a.lse, a.expert_of, a.gate_of}, a.rank_in_block,
                       a.blockcnt, a.partial, [&](int i, int e) { return prob[i * ES + e]; });
}

template <typename XT, int MAXJ>
__global__ __launch_bounds__(kRouterThreads) void router_kernel(
    const XT* __restrict__ x, const float* __restrict__ wr, const float* __restrict__ bias,
    const uint8_t* __restrict__ valid, int T, int d, int E, int k, float* P,
    float* __restrict__ lse, int* __restrict__ expert_of, float* __restrict__ gate_of,
    int* __restrict__ rank_in_block, int* __restrict__ blockcnt, float* __restrict__ partial) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    // (the logits are where the probabilities go: a lane has read its own before it writes them)
    router_tail<MAXJ, kRouterTokens>(lds_raw, blockIdx.x, valid, T, E, k, RouteOut{P, lse, expert_of, gate_of}, rank_in_block, blockcnt,
                                     partial, [&](int i, int e) { return P[((size_t)blockIdx.x * kRouterTokens + i) * E + e]; });
}

// ---------------------------------------------------------------------------
// dispatch_kernel: block b owns the same tokens as router block b.
//
// Prologue (every block, redundantly — the table is a few KB and sits in L2): column sums
// of the per-block histogram give counts[e], their exclusive prefix gives offsets[e], and
// the sums over the blocks before b give this block's base per expert.  Block 0 also
// writes counts / offsets, the tile table of the grouped products (tile i = rows
// [tile_row0[i], tile_row0[i] + tile_rows[i]) of expert tile_expert[i]; a tile never spans
// two experts) and the two auxiliary losses (reference src/moe.rs:602-639), folding the
// per-block partial sums in a fixed order.
//
// Position of a routed slot = offsets[e] + base[e] + rank_in_block[slot]: slots are numbered
// token-major, so this is exactly the order in which the reference appends slots to an
// expert's list (src/moe.rs:266-274).  The optional row copy is `gather_rows`
// (src/moe.rs:658-664); rows move as 16-byte pieces.
// ---------------------------------------------------------------------------
// dispatch_fused_kernel: for a modest number of router blocks the layout scan is folded into the
// dispatch launch: every block re-derives counts, offsets and its own base from all the block
// histograms (O(blocks^2 x experts) reads in total, but one launch less on the critical path);
// block 0 also writes counts, offsets and the tile table, the last block the losses.
size_t dispatch_fused_lds_bytes(int E, int k, int tokens) {
    return layout_lds_bytes(E) + (size_t)tokens * k * 4;
}

template <typename XT>
__global__ __launch_bounds__(256) void dispatch_fused_kernel(
    const XT* __restrict__ x, const int* __restrict__ expert_of, const int* __restrict__ rank_in_block, LayoutArgs l, int d,
    int* __restrict__ perm_slot, int* __restrict__ perm_token, int* __restrict__ inv_pos, XT* __restrict__ xg) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int T = l.T, E = l.E, k = l.k, TB = l.TB;
    int* const lpos = reinterpret_cast<int*>(lds_raw + layout_lds_bytes(E));  // [TB * k]
    const int tid = threadIdx.x;
    const int blk = blockIdx.x;
    // this thread's first slot does not depend on the scan: fetch it before anything else
    const int t0 = blk * TB;
    const int nt = min(TB, T - t0);
    const int nls = nt * k;
    int ex_first = -1, rank_first = 0;
    if (tid < nls) {
        ex_first = expert_of[(size_t)t0 * k + tid];
        rank_first = rank_in_block[(size_t)t0 * k + tid];
    }
    // Block 0 writes counts, offsets and the tile table; the two losses are the work of another block (the last
    // one), so that neither of the two is the launch's long pole.  That block fetches the partial sums in the same
    // batch of loads as the histograms.
    const LayoutSums sums = layout_scan(l, blk, blk == 0, blk == (T + TB - 1) / TB - 1, lds_raw);
    const int* const off = sums.off;
    const int* const base = sums.base;

    for (int ls = tid; ls < nls; ls += 256) {
        const int s = t0 * k + ls;
        const int ex = ls == tid ? ex_first : expert_of[s];
        int pos = -1;
        if (ex >= 0) {
            pos = off[ex] + base[ex] + (ls == tid ? rank_first : rank_in_block[s]);
            perm_slot[pos] = s;
            perm_token[pos] = s / k;
        }
        inv_pos[s] = pos;
        lpos[ls] = pos;
    }
    __syncthreads();
    if (xg == nullptr) return;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    constexpr int VE = 16 / (int)sizeof(XT);  // elements per 16 bytes
    const bool vec = (d % VE == 0);
    for (int ls = wave; ls < nls; ls += 4) {
        const int pos = lpos[ls];
        if (pos < 0) continue;
        const XT* src = x + (size_t)(t0 + ls / k) * d;
        XT* dst = xg + (size_t)pos * d;
        if (vec) {
            const uint4* s4 = reinterpret_cast<const uint4*>(src);
            uint4* d4 = reinterpret_cast<uint4*>(dst);
            for (int c = lane; c < d / VE; c += 64) d4[c] = s4[c];
        } else {
            for (int c = lane; c < d; c += 64) dst[c] = src[c];
        }
    }
}


// layout_columns_kernel: the per-block histograms, a workgroup for every four experts (and the z sums, a column of their
// own): counts and probability masses per expert, and for every router block the number of slots of each expert routed
// by the blocks before it.  The columns share nothing, and what follows from the counts - offsets, tile table, losses - is
// little enough for every block of the dispatch launch to work out for itself.  (One workgroup for everything walked 512
// blocks x 64 experts in 17.6 to 21.8 us; this takes 5.3 to 6.2.)  The blocks are cut into consecutive parts whose
// sums are folded in order.
// router blocks x experts up to which the scan is folded into the dispatch launch instead
constexpr long long kFusedScanLimit = 4096;
constexpr int kColumns = 4;     // experts of a workgroup
constexpr int kColumnParts = 16;

__global__ __launch_bounds__(kColumns * kColumnParts) void layout_columns_kernel(
    const int* __restrict__ blockcnt, const float* __restrict__ partial, int nb, int E, int* __restrict__ blockbase,
    int* __restrict__ counts, float* __restrict__ mass) {
    __shared__ int part_sum[kColumnParts][kColumns];
    __shared__ float part_mass[kColumnParts][kColumns];
    const int c = threadIdx.x % kColumns, p = threadIdx.x / kColumns;
    const int e = blockIdx.x * kColumns + c;  // column E: the z sums; past it: nothing
    const int len = (nb + kColumnParts - 1) / kColumnParts;
    const int b0 = min(nb, p * len), b1 = min(nb, b0 + len);
    const int ec = min(e, E - 1), em = min(e, E);  // (always a valid column: no branch around the loads)
    // Loads come in batches that do not depend on one another: one round trip per batch.  The first kKeep histogram
    // entries of a thread stay in registers for the second pass.
    constexpr int kKeep = 32, kBatch = 16;
    int keep[kKeep];
    int sc = 0;
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < kKeep; i += kBatch) {
        float v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int bb = max(0, min(b0 + i + u, nb - 1));
            keep[i + u] = blockcnt[(size_t)bb * E + ec];
            v[u] = partial[(size_t)bb * (E + 1) + em];
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
            if (b0 + i + u < b1) {
                sc += keep[i + u];
                m += v[u];
            }
    }
    for (int b = b0 + kKeep; b < b1; b += kBatch) {
        int n[kBatch];
        float v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int bb = min(b + u, b1 - 1);
            n[u] = blockcnt[(size_t)bb * E + ec];
            v[u] = partial[(size_t)bb * (E + 1) + em];
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
            if (b + u < b1) {
                sc += n[u];
                m += v[u];
            }
    }
    part_sum[p][c] = sc;
    part_mass[p][c] = m;
    __syncthreads();
    int run = 0, total = 0;
    float all = 0.0f;
    for (int q = 0; q < kColumnParts; ++q) {
        if (q == p) run = total;
        total += part_sum[q][c];
        all += part_mass[q][c];
    }
    if (p == 0) {
        if (e < E) counts[e] = total;
        if (e <= E) mass[e] = all;
    }
    if (e >= E) return;
#pragma unroll
    for (int i = 0; i < kKeep; ++i)
        if (b0 + i < b1) {
            blockbase[(size_t)(b0 + i) * E + e] = run;
            run += keep[i];
        }
    for (int b = b0 + kKeep; b < b1; b += kBatch) {
        int n[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) n[u] = blockcnt[(size_t)min(b + u, b1 - 1) * E + e];
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
            if (b + u < b1) {
                blockbase[(size_t)(b + u) * E + e] = run;
                run += n[u];
            }
    }
}

// Exclusive prefix sum over the 256 threads of a workgroup; `sums`: room for 4 wave totals.
__device__ __forceinline__ int exclusive_prefix_256(int v, int* sums) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(incl, o);
        if (lane >= o) incl += up;
    }
    if (lane == 63) sums[wave] = incl;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int w = 0; w < 3; ++w)
        if (w < wave) before += sums[w];
    return before + incl - v;
}

// ---------------------------------------------------------------------------
// dispatch_kernel: block b owns the same tokens as router block b:
// position = offsets[e] + blockbase[b][e] + rank in block, the offsets being the counts' prefix sums.  Block 0 also
// writes offsets and the tile table, the last block the two auxiliary losses (src/moe.rs:602-639).
// ---------------------------------------------------------------------------
size_t dispatch_lds_bytes(int E, int k, int tokens) {
    return ((size_t)2 * (E + 1) + (size_t)tokens * k) * 4;
}

template <typename XT>
__global__ __launch_bounds__(256) void dispatch_kernel(
    const XT* __restrict__ x, const int* __restrict__ expert_of, const int* __restrict__ rank_in_block,
    const int* __restrict__ blockbase, const int* __restrict__ counts, const float* __restrict__ mass, int T, int d,
    int E, int k, int TB, float w_aux, float w_z, int tile_m, int* __restrict__ offsets, int* __restrict__ tile_expert,
    int* __restrict__ tile_row0, int* __restrict__ tile_rows, int* __restrict__ ntiles, float* __restrict__ losses,
    int* __restrict__ perm_slot, int* __restrict__ perm_token, int* __restrict__ inv_pos, XT* __restrict__ xg) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    int* base = reinterpret_cast<int*>(lds_raw);  // [E+1] slots of each expert routed by earlier blocks
    int* off = base + (E + 1);                    // [E+1] first row of each expert group
    int* lpos = off + (E + 1);                    // [TB * k]

    const int tid = threadIdx.x;
    const int blk = blockIdx.x;
    const int t0 = blk * TB;
    const int nt = min(TB, T - t0);
    const int nls = nt * k;
    // this thread's first slot and the block's two table rows are independent loads
    int ex_first = -1, rank_first = 0;
    if (tid < nls) {
        ex_first = expert_of[(size_t)t0 * k + tid];
        rank_first = rank_in_block[(size_t)t0 * k + tid];
    }
    __shared__ int sums[2][4];
    const int cnt = tid < E ? counts[tid] : 0;  // (at most 256 experts)
    const float ms = mass[min(tid, E)];
    if (tid < E) base[tid] = blockbase[(size_t)blk * E + tid];
    const int first_row = exclusive_prefix_256(cnt, sums[0]);
    if (tid < E) off[tid] = first_row;
    if (tid == E - 1) off[E] = first_row + cnt;
    __syncthreads();
    if (blk == 0) {
        const int n = (cnt + tile_m - 1) / tile_m;
        const int first = exclusive_prefix_256(n, sums[1]);  // its tiles start after those of the experts before it
        if (tid < E) {
            offsets[tid] = first_row;
            for (int i = 0; i < n; ++i) {
                tile_expert[first + i] = tid;
                tile_row0[first + i] = first_row + i * tile_m;
                tile_rows[first + i] = min(tile_m, cnt - i * tile_m);
            }
        }
        if (tid == E - 1) {
            offsets[E] = first_row + cnt;
            ntiles[0] = first + n;
        }
    }
    if (blk == (int)gridDim.x - 1) {
        // every valid token routes exactly k slots, so the valid-token count is routed / k.  The experts' terms (two
        // divisions and a product each) side by side, then their sum in expert order by one thread.
        __shared__ float term[257];
        const int V = off[E] / k;
        const float tokens = (float)V, slots = (float)V * (float)k;
        if (tid < E && V > 0) term[tid] = ((float)cnt / slots) * (ms / tokens);
        if (tid == 0) term[256] = mass[E];
        __syncthreads();
        if (tid == 0) {
            float aux = 0.0f, z = 0.0f;
            if (V > 0) {
                for (int q = 0; q < E; ++q) aux = aux + term[q];
                aux = aux * ((float)E * w_aux);
                z = w_z * term[256] / tokens;
            }
            losses[0] = aux;
            losses[1] = z;
        }
    }

    for (int ls = tid; ls < nls; ls += 256) {
        const int s = t0 * k + ls;
        const int ex = ls == tid ? ex_first : expert_of[s];
        int pos = -1;
        if (ex >= 0) {
            pos = off[ex] + base[ex] + (ls == tid ? rank_first : rank_in_block[s]);
            perm_slot[pos] = s;
            perm_token[pos] = s / k;
        }
        inv_pos[s] = pos;
        lpos[ls] = pos;
    }
    __syncthreads();
    if (xg == nullptr) return;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    constexpr int VE = 16 / (int)sizeof(XT);  // elements per 16 bytes
    const bool vec = (d % VE == 0);
    for (int ls = wave; ls < nls; ls += 4) {
        const int pos = lpos[ls];
        if (pos < 0) continue;
        const XT* src = x + (size_t)(t0 + ls / k) * d;
        XT* dst = xg + (size_t)pos * d;
        if (vec) {
            const uint4* s4 = reinterpret_cast<const uint4*>(src);
            uint4* d4 = reinterpret_cast<uint4*>(dst);
            for (int c = lane; c < d / VE; c += 64) d4[c] = s4[c];
        } else {
            for (int c = lane; c < d; c += 64) dst[c] = src[c];
        }
    }
}

// ---------------------------------------------------------------------------
// combine_kernel: out[t,:] = sum over the token's slots in ascending expert
// order of gate * y[pos,:] (a rounded multiply then a rounded add, as
// src/moe.rs:294-311), then + shared[t,:] (src/moe.rs:313-319), then
// + residual[t,:].  Ascending expert order is ascending position order.
// One thread per (token, 16-byte column piece); the token's slots are sorted
// by position in registers when k <= KMAX (an unused slot is sorted behind them), otherwise found by repeated search.
// ---------------------------------------------------------------------------
// VN consecutive elements of an expert row, as raw bits and widened: the rows are of the layer's activation type, or
// bf16 under f32 activations (a layer whose bf16 / int8 expert products run on the matrix cores).
template <typename YT, typename XT>
struct RowPiece {  // rows of the activation type itself
    typedef uint4 raw_t;
    static __device__ __forceinline__ raw_t load_raw(const YT* p) { return Vec16<YT>::load_raw(p); }
    static __device__ __forceinline__ void widen(const raw_t& a, float (&v)[Vec16<YT>::N]) { Vec16<YT>::widen(a, v); }
};
template <>
struct RowPiece<float, bf16_t> {  // eight f32 elements beside eight bf16 ones
    struct raw_t {
        float4 a, b;
    };
    static __device__ __forceinline__ raw_t load_raw(const float* p) {
        return {*reinterpret_cast<const float4*>(p), *reinterpret_cast<const float4*>(p + 4)};
    }
    static __device__ __forceinline__ void widen(const raw_t& r, float (&v)[8]) {
        v[0] = r.a.x; v[1] = r.a.y; v[2] = r.a.z; v[3] = r.a.w;
        v[4] = r.b.x; v[5] = r.b.y; v[6] = r.b.z; v[7] = r.b.w;
    }
};
template <>
struct RowPiece<bf16_t, float> {  // four bf16 elements beside four f32 ones
    typedef uint2 raw_t;
    static __device__ __forceinline__ raw_t load_raw(const bf16_t* p) { return *reinterpret_cast<const uint2*>(p); }
    static __device__ __forceinline__ void widen(const raw_t& a, float (&v)[4]) {
        v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
        v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
    }
};

// Bound by memory, 268 MB for 16384 tokens of d 1024 with six slots and a shared expert - as long as its vector instructions are
// few: every lane sorting eight (position, gate) pairs by insertion made the kernel 1582 of them long; sorted as a network
// of neighbours, for the least even number of slots, it has 530.
// ROW: a row is whole waves of pieces (d a multiple of 512 in bf16, of 256 in f32), so that a wave's token is known to all its
// lanes, and its positions and gates are fetched and sorted once a wave in scalar registers: 290.  us a forward, before / after: 64
// experts of 704, six a token, d 1024, 16384 rows 673.3 / 665.2 (another box 712.0 / 701.0); 2048 rows of the default model 34.2 /
// 33.9; without whole waves (d 768) 8192 rows by 16 experts, two a token, 147.2 / 146.4, 4096 rows int8 the same.
// PARTS, ROUND: CombineArgs::parts, of rows that are bf16 otherwise.  (What only they need comes last: the others' arguments are one
// cache line.)
template <typename XT, typename YT, int KMAX, bool ROW, int PARTS, bool ROUND>
__global__ __launch_bounds__(256) void combine_vec_kernel(
    const YT* __restrict__ y, const YT* __restrict__ yshared, const XT* __restrict__ residual,
    const int* __restrict__ inv_pos, const float* __restrict__ gate_of, int T, int d, int k, uint32_t recip,
    XT* __restrict__ out, int part_rows, bool shared_in_parts) {
    constexpr int VN = Vec16<XT>::N;
    typedef RowPiece<YT, XT> YP;
    const int pieces = d / VN;
    int t, c;
    if constexpr (ROW) {
        const unsigned wave = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), per = (unsigned)pieces / 64u;
        t = __builtin_amdgcn_readfirstlane((int)(wave / per));
        if (t >= T) return;
        c = (int)((wave - (unsigned)t * per) * 64u + (threadIdx.x & 63)) * VN;
    } else {
        const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
        if (idx >= (long long)T * pieces) return;
        t = recip ? (int)__umulhi((uint32_t)idx, recip) : (int)(idx / pieces);  // (uniform over the launch)
        c = (int)(idx - (long long)t * pieces) * VN;
    }
    // The token's routed slots, sorted by position; those without one (-1) and those past k are the largest numbers.  All are requested
    // before the first is looked at, from addresses that do not depend on one another - a slot past k repeats the last one:
    // loads under a branch would follow one another, two trips to memory a slot in front of the rows'.  (Gates as bits: the
    // compiler chooses between floats in vector registers.)
    uint32_t pos[KMAX], gate[KMAX];
    int n = 0;
#pragma unroll
    for (int r = 0; r < KMAX; ++r) {
        const int rr = r < k ? r : k - 1;
        pos[r] = (uint32_t)inv_pos[(size_t)t * k + rr];
        gate[r] = reinterpret_cast<const uint32_t*>(gate_of)[(size_t)t * k + rr];
    }
#pragma unroll
    for (int r = 0; r < KMAX; ++r) {
        if (r >= k) pos[r] = 0xffffffffu;
        n += (int32_t)pos[r] >= 0 ? 1 : 0;
    }
#pragma unroll
    for (int round = 0; round < KMAX; ++round)  // neighbours in turn
#pragma unroll
        for (int q = round & 1; q + 1 < KMAX; q += 2) {
            // (named values: a choice between array elements would be a choice of an index)
            const uint32_t pa = pos[q], pb = pos[q + 1], ga = gate[q], gb = gate[q + 1];
            const bool swap = pa > pb;
            pos[q] = swap ? pb : pa;
            pos[q + 1] = swap ? pa : pb;
            gate[q] = swap ? gb : ga;
            gate[q + 1] = swap ? ga : gb;
        }
    float acc[VN];
#pragma unroll
    for (int i = 0; i < VN; ++i) acc[i] = 0.0f;
    // every row piece is fetched before the first add (no branch around a load: an unused slot
    // re-reads row 0), so the k loads of a token are one round trip instead of k
    typename YP::raw_t raw[PARTS][KMAX], raw_s[PARTS] = {};
    uint4 raw_r = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int p = 0; p < PARTS; ++p)
#pragma unroll
        for (int r = 0; r < KMAX; ++r) raw[p][r] = YP::load_raw(y + ((size_t)p * part_rows + (r < n ? pos[r] : 0)) * d + c);
    if (yshared) {  // uniform over the launch
#pragma unroll
        for (int p = 0; p < PARTS; ++p)
            if (p == 0 || shared_in_parts) raw_s[p] = YP::load_raw(yshared + ((size_t)p * T + t) * d + c);
    }
    if (residual) raw_r = Vec16<XT>::load_raw(residual + (size_t)t * d + c);
#pragma unroll
    for (int r = 0; r < KMAX; ++r) {
        if (r < n) {
            float v[VN];
            YP::widen(raw[0][r], v);
#pragma unroll
            for (int p = 1; p < PARTS; ++p) {
                float more[VN];
                YP::widen(raw[p][r], more);
#pragma unroll
                for (int i = 0; i < VN; ++i) v[i] = __fadd_rn(v[i], more[i]);
            }
            if constexpr (ROUND)
#pragma unroll
                for (int i = 0; i < VN; ++i) v[i] = to_f32(from_f32<bf16_t>(v[i]));
#pragma unroll
            for (int i = 0; i < VN; ++i) acc[i] = __fadd_rn(acc[i], __fmul_rn(__uint_as_float(gate[r]), v[i]));
        }
    }
    if (yshared) {
        float v[VN];
        YP::widen(raw_s[0], v);
#pragma unroll
        for (int p = 1; p < PARTS; ++p) {
            if (!shared_in_parts) break;
            float more[VN];
            YP::widen(raw_s[p], more);
#pragma unroll
            for (int i = 0; i < VN; ++i) v[i] = __fadd_rn(v[i], more[i]);
        }
        if constexpr (ROUND)
#pragma unroll
            for (int i = 0; i < VN; ++i) v[i] = to_f32(from_f32<bf16_t>(v[i]));
#pragma unroll
        for (int i = 0; i < VN; ++i) acc[i] = __fadd_rn(acc[i], v[i]);
    }
    if (residual) {
        float v[VN];
        Vec16<XT>::widen(raw_r, v);
#pragma unroll
        for (int i = 0; i < VN; ++i) acc[i] = __fadd_rn(acc[i], v[i]);
    }
    Vec16<XT>::store(out + (size_t)t * d + c, acc);
}

// Any k, any d: one wave per token, one column per lane per step.
template <typename XT, typename YT>
__global__ __launch_bounds__(256) void combine_any_kernel(
    const YT* __restrict__ y, const YT* __restrict__ yshared, const XT* __restrict__ residual,
    const int* __restrict__ inv_pos, const float* __restrict__ gate_of, int T, int d, int k,
    XT* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T) return;
    const int* ip = inv_pos + (size_t)t * k;
    const float* gp = gate_of + (size_t)t * k;
    for (int c = lane; c < d; c += 64) {
        float acc = 0.0f;
        int last = -1;
        for (int r = 0; r < k; ++r) {
            int best = 0x7fffffff, bi = -1;  // next smallest position greater than `last`
            for (int q = 0; q < k; ++q) {
                const int p = ip[q];
                if (p > last && p < best) {
                    best = p;
                    bi = q;
                }
            }
            if (bi < 0) break;
            last = best;
            acc = __fadd_rn(acc, __fmul_rn(gp[bi], to_f32(y[(size_t)best * d + c])));
        }
        if (yshared) acc = __fadd_rn(acc, to_f32(yshared[(size_t)t * d + c]));
        if (residual) acc = __fadd_rn(acc, to_f32(residual[(size_t)t * d + c]));
        out[(size_t)t * d + c] = from_f32<XT>(acc);
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// Whether route_fused_kernel takes the call: every expert of a token in one workgroup (at most 64, four per lane),
// rows of whole 8-element pieces on 16-byte boundaries, and a slice of columns that fits LDS.
// Large launches take the two-launch sequence: logits_kernel fetches the router rows with scalar loads and keeps six
// waves on a SIMD, which per (token, expert) pair is the faster arithmetic once the launch fills the chip several
// times over (16 384 tokens x 64 experts: 126 us for both launches against 153 us fused); up to 256 K pairs the
// saved launch and the saved trip of the logits through memory weigh more (8192 x 16: 22 against 25 us).
static int fused_cols(const RouterArgs& a, size_t xsize) {
    if (!a.allow_fused || a.E > 64 || a.d % 8 != 0 || a.d < 8) return 0;
    if ((long long)a.T * a.E > 256 * 1024) return 0;
    if ((reinterpret_cast<uintptr_t>(a.x) & 15) || (reinterpret_cast<uintptr_t>(a.wr) & 15)) return 0;
    if (((size_t)a.d * xsize) % 16 != 0) return 0;
    const int cols = a.E <= 32 ? 256 : 128;
    return fused_lds_bytes(a.E, a.k, cols, xsize) <= 64 * 1024 ? cols : 0;
}

// Whether route_rows_kernel takes the call and with how many tokens a workgroup: the fewest that still give at most one
// workgroup a compute unit (the chain of a workgroup is what a call waits for), more for larger batches.
struct RowsPlan {
    int tokens = 0;  // 0: not taken
    int EG = 0;
    size_t lds = 0;
    int slice = 0;
    bool exact = false;  // route_exact_kernel
};
// Where the other kernels are faster all the same (blocks of 8 tokens never lose).  Times are forwards of narrow experts,
// other kernels / this one.
//   quantized: a dot product is d / 32 steps on 32 threads and the folding of their 32 sums; the shorter the rows and the
//     more products a workgroup has, the more of it is folding, which the kernels with a lane a product
//     (logits_q8_kernel; logits_kernel for bf16 rows) do not have; the line was drawn against the former.
//     16 tokens: d 256, 16 experts 1.03 times as long, 8 experts 0.93; d 384, 32 experts 1.09 / 24 experts 1.00; d 512, 64
//     experts 1.12, 48 experts 1.07 to 0.95; d 768, 64 experts 0.92.  32 tokens: d 256, 8 experts 1.05, 4 experts 0.96; d 384,
//     16 experts 1.14 to 1.03; d 512, 24 experts 1.10 to 1.00, 16 experts 1.06 to 0.97; d 768, 32 experts 1.08 to 0.95.
//   32 tokens, 12 to 24 experts (tiles of 4 x 2): short rows leave too little between the barriers.  bf16 rows, d 256 1.02
//     to 1.04, d 384 0.98 to 1.02; f32 rows, d 512 1.02 to 1.03, d 768 1.00; 8 experts 1.00, 32 experts 0.7 to 1.0.
static bool rows_lose(int d, int E, int tokens, bool quantized, bool f32) {
    if (quantized) return tokens == 16 ? 6 * (E + 28) >= d : 16 * (E + 8) >= d;
    return tokens == 32 && E > 8 && E < 32 && d <= (f32 ? 512 : 256);
}

static size_t rows_lds(const RouterArgs& a, bool exact, int tokens, int EG) {
    const int NL = a.wq ? 32 : 8;
    return exact ? route_exact_lds_bytes(a.E, a.k, a.d, tokens, NL, EG)
                 : route_rows_lds_bytes(a.E, a.k, a.d, tokens, NL, EG, a.norm_w != nullptr);
}

// Calls of more than 16 experts on the matrix cores, which route_exact_kernel takes in any number of rounds otherwise.  Times are
// forwards of experts of 64, this kernel / the others.
//   8 tokens (rows of 2300 elements and more): every router row again for eight tokens, which loses once the logits kernel fills the
//     chip.  d 2560, 32 experts, 9000 rows 169 / 169, 10240 180 / 173, 16384 306 / 267; 64 experts 16384 423 / 387.
//   quantized, 32 tokens: a workgroup's chain is a round of sums for eight experts after the other, one workgroup on a compute unit, and
//     as long whether the launch fills the chip or not.  One round of workgroups: d 256, 64 experts, 4100 rows 50.7 / 45.0, 8192 59.3 /
//     61.8; d 768, 48 experts, 5000 rows 68.4 / 64.1, 5500 69.1 / 71.6; d 1024 74.6 / 71.7, 75.7 / 82.5; d 128, 32 experts 37.7 / 36.4.
//     More: d 256, 32 experts, 9000 rows 61.2 / 49.1; d 512, 17 experts, 16384 rows 88.0 / 81.4; 32 experts, 12000 rows 75.9 / 66.7, 14500
//     81.0 / 84.5, 16384 93.4 / 97.7, 30000 145 / 135; d 768, 12000 rows 95.6 / 86.8, 20000 139 / 133, 24000 150 / 166; d 1024, 12000
//     rows 107 / 100, 20000 163 / 165; d 1280, 9000 rows 117 / 110, 64 experts 127 / 155.
static bool exact_loses(int d, int E, int tokens, int blocks, bool quantized) {
    if (E <= 16) return false;
    if (tokens == kMinRouterTokens) return blocks > 1200;
    if (!quantized || tokens < kRouterTokens) return false;
    if (blocks <= 256) return d < 256 || (E > 32 && 4 * blocks < (d < 768 ? 15 : d < 1024 ? 14 : 12) * E);
    if (d > 1024 && E >= 48) return false;
    const int places = (blocks + 255) / 256 * 256;  // workgroups of that many rounds: an eighth or a fifth of them may be missing
    return d < 512 || E <= 24 || (d < 768 && blocks > 512) || (places - blocks) * (d < 896 ? 8 : 5) > places;
}

static RowsPlan plan_rows(const RouterArgs& a, size_t xsize, bool exact) {
    RowsPlan p;
    const int unit = a.wq ? 32 : 8;  // whole turns of the column lanes, whole 16-byte pieces
    if (!a.allow_fused || a.E > 64 || a.d % unit != 0 || a.d < unit || a.k > kMaxTopK) return p;
    if ((reinterpret_cast<uintptr_t>(a.x) & 15) || ((size_t)a.d * xsize) % 16 != 0) return p;
    if (reinterpret_cast<uintptr_t>(a.wq ? static_cast<const void*>(a.wq) : a.wr) & 15) return p;
    if (a.norm_w && ((reinterpret_cast<uintptr_t>(a.xn_out) & 15) || a.d % 8 != 0)) return p;
    const int NL = a.wq ? 32 : 8;
    p.exact = exact;
    int tokens = a.min_tokens;
    while (tokens < kRouterTokens && (a.T + tokens - 1) / tokens > 256) tokens *= 2;
    for (; tokens >= a.min_tokens && !p.tokens; tokens /= 2) {
        int EG = a.E;  // as many experts' rows as fit together, whole pairs, at least 8 (or all of them)
        auto lds = [&] { return rows_lds(a, p.exact, tokens, EG); };
        const int least = p.exact ? exact_round(tokens, NL) : 8;
        while (EG > least && lds() > (size_t)kMaxRouterLds) EG = p.exact ? exact_fewer(EG, tokens, NL) : (EG - 1) & ~1;
        if (lds() > (size_t)kMaxRouterLds) continue;
        p.tokens = tokens;
        p.EG = EG;
        p.lds = lds();
    }
    if (!p.tokens) return p;
    // Above 256 K pairs: the sequences tuned for launches that fill the chip several times over.  Below, one round of workgroups or
    // none, for the chain of a second round is as long as the first's: 9000 tokens, d 512, 8 experts 60.0 us a forward in two
    // rounds, 57.0 without; 16 experts 63.2 / 57.1, f32 rows 65.8 / 56.7; d 512, 4 experts, two workgroups a unit 55.5 / 61.0.
    // Blocks of 32 tokens lie on a compute unit as its LDS and its registers allow: of route_rows_kernel three up to 8 experts (up to 76
    // registers), two beyond (92); of route_exact_kernel two (106), over a quantized router one (135).  d 256, 8 experts of 64, 20000
    // rows: three of the former 54.7, without 56.8; f32 rows 87.4 / 90.1; short rows the other way round, d 128, 20000 rows 45.5 / 43.8.
    // On the matrix cores a round more all the same where rows are long enough: d 384, 20000 rows 68.0 / 69.6, d 256 57.0 / 54.7, d 128
    // 48.5 / 43.8; quantized, d 512, 8193 rows 47.3 / 50.4, d 256, 12000 rows 51.4 / 49.6.
    const int blocks = (a.T + p.tokens - 1) / p.tokens;
    const int in_lds = (int)((size_t)kMaxRouterLds / p.lds);
    const int a_unit = p.exact ? (a.wq ? (a.d >= 512 ? 2 : 1) : (a.d >= 384 ? 3 : 2)) : (a.wq || a.E > 8 || a.d < 256 ? 2 : 3);
    const int together = p.tokens == kRouterTokens ? 256 * std::min(a_unit, in_lds) : 256;
    // On the matrix cores more than 16 experts in any number of rounds, ahead of a logit a lane and a launch for the rest: us a
    // forward, logits_kernel + router_kernel / route_exact_kernel, 64 experts of 704, d 1024, 16384 rows 672.6 / 651.8, of 64, d 256,
    // 30000 rows 110.0 / 92.3; 32 of 256, d 1024, 9000 rows 121.9 / 111.9, 16384 195.7 / 181.1; of 64, d 2048, 16384 rows 304 / 247 (where
    // not: exact_loses).  Up to 16 experts a chain less per round outweighs it: 16 of 256, d 768, 16384 rows 112.1 / 111.3, quantized
    // 40000 rows 194.7 / 199.3; 8 of 64, d 512, 60000 rows 162.7 / 170.0.
    // So do f32 rows on the vector units: a thread's tile of tokens and experts reads LDS once for several products, where the other
    // kernels read it for each and take the rows once for every eight experts.  us a forward, experts of 64, the others / this one:
    // d 256, 32 experts, 8500 rows 64.5 / 52.3, 30000 128 / 90; 64 experts, 4500 rows 62.1 / 50.2, 8192 82.8 / 54.7; d 512, 32 experts,
    // 8500 rows 94.6 / 71.2, 48 experts, 16384 160 / 113; d 768, 32 experts, 12000 rows 137 / 108, 64 experts, 8192 170 / 92; d 1024, 32
    // experts, 4500 rows 115 / 82, 64 experts, 16384 337 / 248; d 2048, 32 experts, 12000 rows 316 / 308; quantized, d 768, 32 experts,
    // 16384 rows 184 / 155, d 1024, 64 experts, 8500 rows 220 / 164.  Not where route_fused_kernel has the rows (up to 26 experts and 256 K
    // pairs): d 768, 20 experts, 12000 rows 93.5 / 97.4, d 1024, 24 experts, 8500 rows 105 / 113, d 512, 22 experts, 10500 rows 67.7 / 71.4, d 128,
    // 20 experts, 8500 rows 39.1 / 40.7; without it d 128, 28 experts, 4200 rows 41.7 / 36.9, d 512, 31 experts 74.9 / 52.9, 24 experts, 12000
    // rows 98.3 / 75.2, d 64, 24 experts, 16384 and 20000 rows 45.5 / 43.0, 52.7 / 54.2.  Under a quantized router there too, d 640, 24
    // experts, 8300 rows 94.1 / 84.8, d 1280, 17 experts, 5000 rows 99.2 / 89.3, but not in little more than one round of workgroups of which
    // a unit takes one: d 768, 20 and 28 experts, 9000 rows 95.3 / 102.2, 105.5 / 114.5, d 896, 30 experts, 8300 rows 122 / 128 (d 896, 20
    // experts, 10500 rows 129 / 118).  Up to 16 experts as above: d 768, 16 experts, 16384 rows 123 / 133.
    const bool any_f32 = !p.exact && xsize == 4 && a.E > 16 && (a.wq || fused_cols(a, xsize) == 0);
    const bool any_size = (p.exact && a.E > 16) || any_f32;
    if (!any_size && ((long long)a.T * a.E > 256 * 1024 || blocks > together)) p.tokens = 0;
    if (p.exact && exact_loses(a.d, a.E, p.tokens, blocks, a.wq != nullptr)) p.tokens = 0;
    // (over f32 rows without a quantized router rows_lose's lines are drawn against route_fused_kernel)
    if (p.tokens > kMinRouterTokens && !p.exact && !(any_f32 && !a.wq) && rows_lose(a.d, a.E, p.tokens, a.wq != nullptr, xsize == 4))
        p.tokens = 0;
    // In several rounds a workgroup's loads, sums and softmax follow one another with nothing beside them where it fills a compute
    // unit's LDS by itself.  So blocks and router rows are made smaller until two lie there together, if they can be: experts past
    // those whose rows lie in LDS follow through the place of the ones before, and blocks of 16 tokens take the router's rows twice as
    // often, which is the smaller loss; and beside a shared expert's products there is room for one of their workgroups.  us a
    // forward, experts of 64, one workgroup a unit / two: blocks of 32, d 512, 32 experts, 8200, 12000, 20000 rows 54.8 / 48.4, 61.5 / 55.5,
    // 93.1 / 83.8, 64 experts 67.6 / 59.4, 75.2 / 67.0, 115 / 104; of 16, d 768, 24 experts 63.1 / 59.2, 77.6 / 71.3, 114 / 106, d 1024,
    // 32 experts 75.7 / 72.9, 93.1 / 87.1, 139 / 130, 64 experts 101 / 91, 115 / 105, 172 / 156; quantized, d 512, 48 experts, 16384 rows
    // 104 / 91; 64 experts of 704, six a row, and a shared one, d 1024, 16384 rows 658 / 648.  (In one round, 5000 rows: 1 to 2 %,
    // not taken; narrower rows lie there twice as they are, wider ones do not fit.)
    // f32 rows: d 256, 48 experts, 12000 rows 72.6 / 66.2; d 512, 17 and 32 experts, 8500 rows 74.4 / 64.4, 77.8 / 72.4; d 768, 40 experts 107 / 102;
    // d 1024, 64 experts, 8500, 16384 rows 183 / 165, 257 / 255.  The gain is the last round's, which two workgroups beside one another make
    // shorter.  Where that is more than half full and half as large blocks take the router's rows in twice as many groups, there is none: d 512,
    // 40 experts, 13000 and 16384 rows (1.6 and 2 rounds) 94.1 / 97.1, 107.4 / 110.8, but 10240 (1.25) 89.1 / 85.1; d 768, 48 experts, 13000 rows
    // 128.5 / 134.9; d 1024, 32 experts, 12000, 15500, 20000 rows (2.9, 3.8, 4.9) 143.8 / 149.5, 177.5 / 185.9, 216.5 / 225.9, 13000 (3.2) 165.6 /
    // 162.6 (40 experts, in whole groups, 2 to 3 % faster all the same, not taken: 20000 rows 243 / 236).  A quantized router's sums take longer
    // than its rows: d 512, 40 experts, 16384 rows 140 / 135, d 1024, 32 experts 202 / 194.
    if (((p.exact && p.tokens == kRouterTokens) || (any_f32 && p.tokens)) && blocks > 256 && p.lds > (size_t)kMaxRouterLds / 2)
        for (int t = p.tokens; t >= std::max(a.min_tokens, p.tokens / 2); t /= 2) {
            const int least = p.exact ? exact_round(t, NL) : 8;
            int EG = a.E;
            while (EG > least && rows_lds(a, p.exact, t, EG) > (size_t)kMaxRouterLds / 2)
                EG = p.exact ? exact_fewer(EG, t, NL) : (EG - 1) & ~1;
            if (rows_lds(a, p.exact, t, EG) > (size_t)kMaxRouterLds / 2) continue;
            auto groups = [&](int eg) { return (a.E + eg - 1) / eg; };
            if (any_f32 && !a.wq && t < p.tokens && (blocks - 1) % 256 >= 128 && groups(EG) >= 2 * groups(p.EG)) continue;
            p.tokens = t;
            p.EG = EG;
            p.lds = rows_lds(a, p.exact, t, EG);
            break;
        }
    if (any_f32 && a.wq && p.tokens && blocks > 256 && blocks <= 320 && p.lds > (size_t)kMaxRouterLds / 2 && fused_cols(a, xsize) != 0) p.tokens = 0;
    // A few tokens by many experts: one workgroup a block would take the experts' rows through its own LDS one group after the
    // other (64 experts of d 1024: 27 us, whatever the tokens).  So the block's experts are shared out, eight to a workgroup
    // or as many as leave at most one round of workgroups; the last to arrive does the rest.  us a forward, one workgroup / shared
    // out: 64 experts, d 1024, 1 row 52.5 / 40.2, 256 rows 100.7 / 87.4, 512 rows 106.3 / 93.9; 32 experts, d 1024, f32, 24 rows
    // 59.6 / 53.7; d 768 38.2 / 36.4; d 512, 128 rows 34.4 / 33.2, but d 256, 128 rows 27.1 / 27.2, 512 rows 29.1 / 29.5; 16 experts,
    // d 768, 64 rows 38.4 / 39.2.
    if (p.tokens == kMinRouterTokens && a.arrive && a.E >= 32 && a.E * a.d >= 16 * 1024)
        for (int slice = 8; slice < a.E && !p.slice; slice *= 2)
            if (blocks * ((a.E + slice - 1) / slice) <= 256) {
                p.slice = slice;
                p.EG = std::min(p.EG, slice);
                p.lds = rows_lds(a, p.exact, p.tokens, p.EG);
            }
    return p;
}

RouterPlan plan_router(const RouterArgs& a, bool bf16) {
    RowsPlan p = plan_rows(a, bf16 ? 2 : 4, route_exact_ok(a, bf16));
    if (!p.tokens && p.exact) p = plan_rows(a, bf16 ? 2 : 4, false);
    RouterPlan q;
    q.block_tokens = p.tokens ? p.tokens : kRouterTokens;
    q.row_experts = p.tokens ? p.EG : 0;
    q.row_lds = p.tokens ? p.lds : 0;
    q.row_slice = p.tokens ? p.slice : 0;
    q.row_exact = p.tokens && p.exact;
    // where the squares' room costs tokens a workgroup, a second round of workgroups costs more than the norm in a launch of
    // its own (8192 tokens, d 768, squares in LDS: 37.7 us in two rounds, 16.2 + 8 in two launches; a wave a row leaves one
    // round: 29 in one launch, 12.5 + 20 in two)
    q.takes_norm = a.norm_w && p.tokens && (a.T + p.tokens - 1) / p.tokens <= 256;
    q.q8_writes_rows16 = p.tokens != 0;
    return q;
}

RouterPlan plan_router_behind_norm(RouterArgs& a, const void* normed, bool bf16, bool* norm_apart) {
    const RouterPlan p = plan_router(a, bf16);
    *norm_apart = a.norm_w && !p.takes_norm;
    if (!*norm_apart) return p;
    a.x = normed;
    a.norm_w = nullptr;
    a.xn_out = nullptr;
    return plan_router(a, bf16);
}

bool router_takes(const RouterArgs& a, const RouterPlan& p, bool bf16) {
    return p == plan_router(a, bf16) && (!a.norm_w || p.takes_norm);
}

template <typename XT>
static hipError_t launch_rows_t(const RouterArgs& a, const RouterPlan& p, hipStream_t s) {
    RouteRowsArgs r{a.x, a.wr, a.wq, a.wscale, a.bias, a.valid, a.T, a.d, a.E, a.k, p.row_experts, a.P, a.lse, a.expert_of, a.gate_of,
                    a.rank_in_block, a.blockcnt, a.partial, static_cast<bf16_t*>(a.rows16), a.norm_w, a.norm_eps, a.xn_out,
                    false, p.row_slice, a.arrive};
    const dim3 grid((a.T + p.block_tokens - 1) / p.block_tokens, p.row_slice ? (a.E + p.row_slice - 1) / p.row_slice : 1);
    auto go = [&](auto kernel) -> hipError_t {
        static std::atomic<unsigned long long> attr_set{0};  // one per kernel: the lambda's body is instantiated for each
        const hipError_t e = once_per_device(attr_set, [&] {
            return hipFuncSetAttribute(reinterpret_cast<const void*>(+kernel.value), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       kMaxRouterLds);
        });
        if (e != hipSuccess) return e;
        RB_LAUNCH(kernel.value, grid, dim3(kRouterThreads), p.row_lds, s, r);
        return hipGetLastError();
    };
#define RB_ROUTE_ROWS(TB, NL, TT, EE)                                                                                    \
    (a.norm_w ? go(std::integral_constant<void (*)(RouteRowsArgs), &route_rows_kernel<XT, TB, NL, TT, EE, true>>{})     \
              : go(std::integral_constant<void (*)(RouteRowsArgs), &route_rows_kernel<XT, TB, NL, TT, EE, false>>{}))
    // tokens x experts a thread: the largest tile that still has work for every thread (more sums a thread mean less
    // traffic with LDS; the sums of 8 tokens x 16 experts take 2.3 us with 1 x 2 on eight waves, 2.9 with 2 x 2 on four)
    if (a.wq) {
        if (p.block_tokens == 8) return RB_ROUTE_ROWS(8, 32, 2, 2);
        if (p.block_tokens == 16) return RB_ROUTE_ROWS(16, 32, 4, 2);
        return RB_ROUTE_ROWS(32, 32, 4, 2);
    }
    if (p.block_tokens == 8) return RB_ROUTE_ROWS(8, 8, 1, 2);
    if (p.block_tokens == 16) return a.E <= 8 ? RB_ROUTE_ROWS(16, 8, 1, 2) : RB_ROUTE_ROWS(16, 8, 2, 2);
    return a.E <= 8 ? RB_ROUTE_ROWS(32, 8, 2, 2) : RB_ROUTE_ROWS(32, 8, 4, 2);
#undef RB_ROUTE_ROWS
}

template <typename XT>
static hipError_t launch_router_t(const RouterArgs& a, const RouterPlan& p, hipStream_t s) {
    if (p.row_exact) return launch_route_exact(a, p, s);
    if (p.row_experts) return launch_rows_t<XT>(a, p, s);
    const int nb = (a.T + kRouterTokens - 1) / kRouterTokens;
    if (const int cols = a.wq ? 0 : fused_cols(a, sizeof(XT))) {
        // bf16 rows staged as f32 where a slice of the same width then still fits
        const bool wide = sizeof(XT) == 2 && fused_cols(a, 4) == cols;
        const size_t lds = fused_lds_bytes(a.E, a.k, cols, wide ? 4 : sizeof(XT));
        auto go = [&](auto ni, auto wide_tag) {
            RB_LAUNCH((route_fused_kernel<XT, decltype(ni)::value, decltype(wide_tag)::value>), dim3(nb),
                               dim3(kRouterThreads), lds, s,
                               static_cast<const XT*>(a.x), a.wr, a.bias, a.valid, a.T, a.d, a.E, a.k, cols, a.P, a.lse,
                               a.expert_of, a.gate_of, a.rank_in_block, a.blockcnt, a.partial,
                               static_cast<bf16_t*>(a.rows16));
        };
        auto pick = [&](auto wide_tag) {
            if (a.E <= 16) go(std::integral_constant<int, 1>{}, wide_tag);
            else if (a.E <= 32) go(std::integral_constant<int, 2>{}, wide_tag);
            else go(std::integral_constant<int, 4>{}, wide_tag);
        };
        if constexpr (sizeof(XT) == 2) {
            if (wide) pick(std::true_type{});
            else pick(std::false_type{});
        } else {
            pick(std::false_type{});
        }
        return hipGetLastError();
    }
    static std::atomic<unsigned long long> attr_set{0};
    {  // allow more than the default 64 KiB of dynamic LDS (gfx950 has 160 KiB per CU)
        const hipError_t e = once_per_device(attr_set, [] {
            hipError_t r = hipFuncSetAttribute(reinterpret_cast<const void*>(router_kernel<XT, 1>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kMaxRouterLds);
            if (r == hipSuccess)
                r = hipFuncSetAttribute(reinterpret_cast<const void*>(router_kernel<XT, kMaxExperts / 64>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, kMaxRouterLds);
            return r;
        });
        if (e != hipSuccess) return e;
    }
    // eight experts (waves) per workgroup share one staged slice of 64 token rows
    constexpr int NE = 8;
    const int tiles_t = (a.T + kLogitTokens - 1) / kLogitTokens;
    const dim3 lgrid(tiles_t, (a.E + NE - 1) / NE);
    if (a.wq && (a.rows16 || !a.wscale)) return hipErrorInvalidValue;  // (the caller casts f32 rows itself on this path)
    auto logits = [&](auto lanes) {
        constexpr int NL = decltype(lanes)::value;
        if ((long long)lgrid.x * lgrid.y <= 512)  // at most two workgroups on a compute unit
            RB_LAUNCH((logits_kernel<XT, NE, true, false, NL>), lgrid, dim3(NE * 64), 0, s, static_cast<const XT*>(a.x),
                      a.wr, a.bias, a.T, a.d, a.E, a.P, static_cast<bf16_t*>(a.rows16), a.wscale);
        else
            RB_LAUNCH((logits_kernel<XT, NE, false, sizeof(XT) == 2, NL>), lgrid, dim3(NE * 64), 0, s,
                      static_cast<const XT*>(a.x), a.wr, a.bias, a.T, a.d, a.E, a.P, static_cast<bf16_t*>(a.rows16), a.wscale);
    };
    if (!a.wq) {
        logits(std::integral_constant<int, 8>{});
    } else if constexpr (sizeof(XT) == 2) {
        logits(std::integral_constant<int, 32>{});
    } else {
        const long long pairs = (long long)a.T * a.E;
        RB_LAUNCH(logits_q8_kernel<XT>, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, s,
                  static_cast<const XT*>(a.x), a.wq, a.wscale, a.bias, a.T, a.d, a.E, a.P);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (a.E <= 64)
        RB_LAUNCH((router_kernel<XT, 1>), dim3(nb), dim3(kRouterThreads), router_lds_bytes(a.E, a.k), s,
                           static_cast<const XT*>(a.x), a.wr, a.bias, a.valid, a.T, a.d, a.E, a.k, a.P, a.lse,
                           a.expert_of, a.gate_of, a.rank_in_block, a.blockcnt, a.partial);
    else
        RB_LAUNCH((router_kernel<XT, kMaxExperts / 64>), dim3(nb), dim3(kRouterThreads),
                           router_lds_bytes(a.E, a.k), s, static_cast<const XT*>(a.x), a.wr, a.bias, a.valid, a.T, a.d,
                           a.E, a.k, a.P, a.lse, a.expert_of, a.gate_of, a.rank_in_block, a.blockcnt, a.partial);
    return hipGetLastError();
}

hipError_t launch_router(const RouterArgs& a, const RouterPlan& p, bool bf16, hipStream_t s) {
    if (a.T <= 0) return hipSuccess;
    if (!router_takes(a, p, bf16)) return hipErrorInvalidValue;  // (its blocks would not be those the dispatch counts)
    if (a.rows16 && (bf16 || a.d % 8 != 0)) return hipErrorInvalidValue;  // the copy rides on the 8-element pieces
    return bf16 ? launch_router_t<bf16_t>(a, p, s) : launch_router_t<float>(a, p, s);
}

static LayoutArgs layout_args(const DispatchArgs& a) {
    return {a.blockcnt, a.partial, a.T, a.E, a.k, a.block_tokens, a.w_aux, a.w_z, a.tile_m, a.counts, a.offsets,
            a.tile_expert, a.tile_row0, a.tile_rows, a.ntiles, a.losses};
}

bool dispatch_in_product_ok(const DispatchArgs& a) {
    if (a.T <= 0 || a.xg != nullptr || a.E > 64 || (a.E & (a.E - 1)) != 0) return false;
    const long long nb = (a.T + a.block_tokens - 1) / a.block_tokens;
    return nb * a.E <= kSlotsMaxHistogram && nb <= kSlotsMaxBlocks && (a.block_tokens & (a.block_tokens - 1)) == 0 &&
           (a.tile_m & (a.tile_m - 1)) == 0 && a.tile_m <= kSlotsTileM;
}
RoutedSlots routed_slots(const DispatchArgs& a) {
    RoutedSlots r;
    r.expert_of = a.expert_of;
    r.rank_in_block = a.rank_in_block;
    r.perm_slot = a.perm_slot;
    r.perm_token = a.perm_token;
    r.inv_pos = a.inv_pos;
    r.k_recip = (uint32_t)(0x100000000ull / (uint32_t)a.k) + 1u;
    for (int tb = a.block_tokens; tb > 1; tb >>= 1) ++r.tb_shift;
    for (int m = a.tile_m; m > 1; m >>= 1) ++r.tile_shift;
    r.layout = layout_args(a);
    return r;
}

template <typename XT>
static hipError_t launch_dispatch_t(const DispatchArgs& a, hipStream_t s) {
    const int nb = (a.T + a.block_tokens - 1) / a.block_tokens;
    if ((long long)nb * a.E <= kFusedScanLimit) {
        RB_LAUNCH(dispatch_fused_kernel<XT>, dim3(nb > 0 ? nb : 1), dim3(256),
                           dispatch_fused_lds_bytes(a.E, a.k, a.block_tokens), s, static_cast<const XT*>(a.x), a.expert_of,
                           a.rank_in_block, layout_args(a), a.d, a.perm_slot, a.perm_token, a.inv_pos, static_cast<XT*>(a.xg));
        return hipGetLastError();
    }
    float* const mass = reinterpret_cast<float*>(a.blockbase + (size_t)nb * a.E);  // [E + 1]
    RB_LAUNCH(layout_columns_kernel, dim3(a.E / kColumns + 1), dim3(kColumns * kColumnParts), 0, s, a.blockcnt, a.partial, nb,
              a.E, a.blockbase, a.counts, mass);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    RB_LAUNCH(dispatch_kernel<XT>, dim3(nb), dim3(256), dispatch_lds_bytes(a.E, a.k, a.block_tokens), s,
              static_cast<const XT*>(a.x), a.expert_of, a.rank_in_block, a.blockbase, a.counts, mass, a.T, a.d, a.E, a.k,
              a.block_tokens, a.w_aux, a.w_z, a.tile_m, a.offsets, a.tile_expert, a.tile_row0, a.tile_rows, a.ntiles,
              a.losses, a.perm_slot, a.perm_token, a.inv_pos, static_cast<XT*>(a.xg));
    return hipGetLastError();
}

hipError_t launch_dispatch(const DispatchArgs& a, bool bf16, hipStream_t s) {
    return bf16 ? launch_dispatch_t<bf16_t>(a, s) : launch_dispatch_t<float>(a, s);
}

template <typename XT, typename YT, bool ROUND = false>
static hipError_t launch_combine_t(const CombineArgs& a, hipStream_t s) {
    const YT* y = static_cast<const YT*>(a.y);
    const YT* ys = static_cast<const YT*>(a.yshared);
    const XT* res = static_cast<const XT*>(a.residual);
    XT* out = static_cast<XT*>(a.out);
    constexpr int VN = Vec16<XT>::N;
    const bool pieces_ok = a.d % VN == 0 && a.k <= 8;
    if (a.parts != 1 && (!pieces_ok || sizeof(YT) != 4 || (a.parts != 2 && a.parts != 4))) return hipErrorInvalidValue;
    if (ROUND && (a.parts == 1 || (ys && !a.shared_in_parts))) return hipErrorInvalidValue;  // (rows that are not in parts are bf16)
    if (pieces_ok) {
        const long long total = (long long)a.T * (a.d / VN);
        const dim3 grid((unsigned)((total + 255) / 256)), block(256);
        // 2^32 / pieces rounded up, which counts a row's pieces exactly as long as threads x pieces stays below 2^32 (0: divide)
        const int pieces = a.d / VN;
        const uint32_t recip = pieces > 1 && (total + 256) * pieces < (1ll << 32) ? (uint32_t)(0x100000000ull / (uint32_t)pieces) + 1u : 0u;
        auto launch = [&](auto kmax, auto row, auto parts) {
            RB_LAUNCH((combine_vec_kernel<XT, YT, decltype(kmax)::value, decltype(row)::value, decltype(parts)::value, ROUND>), grid,
                      block, 0, s, y, ys, res, a.inv_pos, a.gate_of, a.T, a.d, a.k, recip, out, a.part_rows, a.shared_in_parts);
        };
        auto go = [&](auto kmax, auto row) {
            if constexpr (sizeof(YT) == 4) {
                if (a.parts == 4) return launch(kmax, row, std::integral_constant<int, 4>{});
                if (a.parts == 2) return launch(kmax, row, std::integral_constant<int, 2>{});
            }
            if constexpr (!ROUND) launch(kmax, row, std::integral_constant<int, 1>{});
        };
        auto pick = [&](auto row) {
            if (a.k <= 2) go(std::integral_constant<int, 2>{}, row);
            else if (a.k <= 4) go(std::integral_constant<int, 4>{}, row);
            else if (a.k <= 6) go(std::integral_constant<int, 6>{}, row);
            else go(std::integral_constant<int, 8>{}, row);
        };
        // (waves are counted in 32 bits)
        if (a.d / VN % 64 == 0 && total / 64 < (1ll << 31)) pick(std::true_type{});
        else pick(std::false_type{});
    } else if constexpr (!ROUND) {
        RB_LAUNCH((combine_any_kernel<XT, YT>), dim3((a.T + 3) / 4), dim3(256), 0, s, y, ys, res, a.inv_pos,
                           a.gate_of, a.T, a.d, a.k, out);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// RmsNorm::forward (src/norm.rs:41-61, inverse_rms :128-131) in front of the layer
// (feed_forward_norm, src/transformer_block.rs:216).  The sum of squares of a row is the
// reference's sequential f32 sum in index order, so the normed rows (and with them the routing)
// come out identical; the output is (value * inverse_rms) * weight, two separately rounded
// products as in the reference.
//
// The chain of d dependent additions per row is the floor of this kernel (2.6 us for 768 columns).  To keep everything
// else off that chain, a block copies its R rows into LDS with every lane's loads in flight at once (the rows of a block
// are one contiguous range) and lays their squares beside them, lane r of the first wave adds up the squares of row r,
// then the whole block writes the normed rows from the LDS copy - the input is read from memory once.
// ---------------------------------------------------------------------------
template <typename XT>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const XT* __restrict__ x, const float* __restrict__ weight,
                                                           float eps, int T, int d, int R, XT* __restrict__ out) {
    constexpr int VN = Vec16<XT>::N;
    extern __shared__ __attribute__((aligned(16))) char smem[];  // R rows, R rows of squares d + 4 floats apart, 256 bytes
    XT* const rows = reinterpret_cast<XT*>(smem);
    float* const sq = reinterpret_cast<float*>(smem + (((size_t)R * d * sizeof(XT) + 15) & ~(size_t)15));
    const int sp = d + 4;
    const int tid = threadIdx.x;
    const int row0 = blockIdx.x * R;
    const int nrows = min(R, T - row0);
    const int pieces = d / VN;  // d is a multiple of 8 (checked by the launcher)
    const uint32_t recip = (uint32_t)(0x100000000ull / (uint32_t)pieces) + 1u;  // idx / pieces, exact for a block's few thousand
    const XT* const src = x + (size_t)row0 * d;
#pragma unroll 4
    for (int idx = tid; idx < nrows * pieces; idx += 256) {
        const int r = pieces == 1 ? idx : (int)__umulhi((uint32_t)idx, recip), p = idx - r * pieces;
        const uint4 raw = *reinterpret_cast<const uint4*>(src + (size_t)idx * VN);
        *reinterpret_cast<uint4*>(rows + (size_t)idx * VN) = raw;
        float v[VN];
        Vec16<XT>::widen(raw, v);
        float4* const s4 = reinterpret_cast<float4*>(sq + r * sp + p * VN);
#pragma unroll
        for (int q = 0; q < VN / 4; ++q)
            s4[q] = make_float4(__fmul_rn(v[4 * q], v[4 * q]), __fmul_rn(v[4 * q + 1], v[4 * q + 1]),
                                __fmul_rn(v[4 * q + 2], v[4 * q + 2]), __fmul_rn(v[4 * q + 3], v[4 * q + 3]));
    }
    __syncthreads();
    if (tid < nrows) {
        const float f = inverse_rms_of(ordered_sum(sq + tid * sp, d), d, eps);
        sq[tid * sp] = f;  // (the row's squares are used up)
    }
    __syncthreads();
    XT* const dst = out + (size_t)row0 * d;
    for (int idx = tid; idx < nrows * pieces; idx += 256) {
        const int r = pieces == 1 ? idx : (int)__umulhi((uint32_t)idx, recip), p = idx - r * pieces;
        float v[VN], o[VN];
        Vec16<XT>::load(rows + (size_t)idx * VN, v);
        const float s = sq[r * sp];
        const float4* w = reinterpret_cast<const float4*>(weight + p * VN);
#pragma unroll
        for (int q = 0; q < VN / 4; ++q) {
            const float4 wv = w[q];
            o[4 * q + 0] = __fmul_rn(__fmul_rn(v[4 * q + 0], s), wv.x);
            o[4 * q + 1] = __fmul_rn(__fmul_rn(v[4 * q + 1], s), wv.y);
            o[4 * q + 2] = __fmul_rn(__fmul_rn(v[4 * q + 2], s), wv.z);
            o[4 * q + 3] = __fmul_rn(__fmul_rn(v[4 * q + 3], s), wv.w);
        }
        Vec16<XT>::store(dst + (size_t)idx * VN, o);
    }
}

// Any width, rows straight from memory: one thread per row for the sum, then the block walks its 64 rows.
template <typename XT>
__global__ __launch_bounds__(64) void rmsnorm_rows_direct_kernel(const XT* __restrict__ x,
                                                                 const float* __restrict__ weight, float eps, int T,
                                                                 int d, XT* __restrict__ out) {
    __shared__ float inv[64];
    const int lane = threadIdx.x;
    const int row0 = blockIdx.x * 64;
    const int my = min(row0 + lane, T - 1);  // rows past the end: a valid row, result unused
    const XT* xr = x + (size_t)my * d;
    float sum = 0.0f;
    for (int c = 0; c < d; ++c) {
        const float v = to_f32(xr[c]);
        sum = __fadd_rn(sum, __fmul_rn(v, v));
    }
    inv[lane] = inverse_rms_of(sum, d, eps);
    __syncthreads();
    const int nrows = min(64, T - row0);
    for (int idx = lane; idx < nrows * d; idx += 64) {
        const int r = idx / d, c = idx - r * d;
        const float v = to_f32(x[(size_t)(row0 + r) * d + c]);
        out[(size_t)(row0 + r) * d + c] = from_f32<XT>(__fmul_rn(__fmul_rn(v, inv[r]), weight[c]));
    }
}

template <typename XT>
hipError_t launch_rmsnorm_t(const XT* x, const float* weight, float eps, int T, int d, XT* out, hipStream_t s) {
    const bool pieces_ok = d % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
                           (reinterpret_cast<uintptr_t>(out) & 15) == 0 && (reinterpret_cast<uintptr_t>(weight) & 15) == 0;
    auto lds_of = [&](int R) { return (((size_t)R * d * sizeof(XT) + 15) & ~(size_t)15) + (size_t)R * (d + 4) * 4 + 256; };
    // rows a block: few enough that the rows' chains spread over the chip (the chain of one row is the time of a small
    // call), enough blocks a compute unit for the loads of one to cover the chain of another (a chain a lane is fewer
    // instructions a row than ordered_sum_wave: 16384 rows, d 768 19 us, a wave a row 27)
    if (pieces_ok && lds_of(1) <= 64 * 1024) {
        int R = std::max(1, std::min(16, (T + 1023) / 1024));
        while (R > 1 && lds_of(R) > 40 * 1024) --R;
        RB_LAUNCH(rmsnorm_rows_kernel<XT>, dim3((T + R - 1) / R), dim3(256), lds_of(R), s, x, weight, eps, T, d, R, out);
    } else {
        RB_LAUNCH(rmsnorm_rows_direct_kernel<XT>, dim3((T + 63) / 64), dim3(64), 0, s, x, weight, eps, T, d,
                           out);
    }
    return hipGetLastError();
}

hipError_t launch_rmsnorm(const void* x, const float* weight, float eps, int T, int d, void* out, bool bf16,
                          hipStream_t s) {
    if (T <= 0) return hipSuccess;
    return bf16 ? launch_rmsnorm_t(static_cast<const bf16_t*>(x), weight, eps, T, d, static_cast<bf16_t*>(out), s)
                : launch_rmsnorm_t(static_cast<const float*>(x), weight, eps, T, d, static_cast<float*>(out), s);
}

hipError_t launch_combine(const CombineArgs& a, bool bf16, hipStream_t s) {
    if (a.T <= 0) return hipSuccess;
    if (a.parts > 1 && (bf16 || a.rows_bf16))
        return bf16 ? launch_combine_t<bf16_t, float, true>(a, s) : launch_combine_t<float, float, true>(a, s);
    if (bf16) return launch_combine_t<bf16_t, bf16_t>(a, s);
    return a.rows_bf16 ? launch_combine_t<float, bf16_t>(a, s) : launch_combine_t<float, float>(a, s);
}

}  // namespace rbmoe
