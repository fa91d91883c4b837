// Grouped expert products on the bf16 matrix cores of gfx950.
//
//   out[row, n] = sum_c a[row, c] * w[expert][n, c]                 (down product)
//   out[row, n] = silu(a . wgate[n]) * (a . wup[n])                 (gate/up product)
//
// Data paths (nothing is staged through registers on its way to LDS):
//   weights      packed at upload into matrix-core operand order (see
//                pack_weight_bf16 / pack_weight_i8); every wave streams its own
//                fragments global -> VGPR through a 4-deep register ring, i.e.
//                the load for reduction step g + 3 is issued while step g runs.
//                int8 weights are widened to bf16 in registers during the step
//                before their multiplies; the per-row scale multiplies the
//                accumulator.
//   activations  128 token rows per workgroup, 160 in tall tiles (gathered through
//                an index for the gate/up product) go global -> LDS with the LDS-DMA load
//                (global_load_lds_dwordx4): lane l of a wave deposits its 16
//                bytes at LDS base + 16 l, so the XOR swizzle that keeps the
//                fragment reads free of bank conflicts is applied by choosing
//                which global piece each lane fetches.  Three LDS stages: the
//                DMA for slice k + 2 is issued in the last step of slice k, after
//                the barrier (behind step KS - 2) that proves its stage free, and
//                is awaited (vmcnt) just before the barrier of slice k + 1.
//   fragments    token fragments are read from LDS one step ahead of the
//                multiplies that use them, across slice boundaries too.
//   issue order  a wave that is alone on its SIMD must keep the matrix core fed
//                by itself: every memory instruction of the main loop sits
//                behind a multiply of its own (see pipe_loop).
// A workgroup is 4 waves side by side along the output features; a wave owns
// all its tokens x 64 weight rows (32 gate + the matching 32 up rows, or 64 down
// rows).  The weight fragment is the matrix-core A operand and the token
// fragment the B operand, so a lane ends with 4 consecutive output features of
// one token and writes them with one 8-byte store.  Token blocks of 32 rows
// that lie beyond the end of a group are skipped, so a ragged group costs at
// most 31 rows of padding.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "layout_device.h"
#include "rbmoe_kernels.h"

// Hook for timeline studies of the kernels: a harness that includes this file may define it to record a time
// stamp per tile (`slot` = the tile's number in launch order) at point i (0 tile taken up, 1 main loop entered,
// 2 main loop left, 3 tile written).  Expands to nothing in the library.
#ifndef RBMOE_TRACE_AT
#define RBMOE_TRACE_AT(slot, i)
#endif

namespace rbmoe {

namespace {

#ifndef RBMOE_STREAM_OCC
#define RBMOE_STREAM_OCC 2
#endif
constexpr int BK = 64;    // reduction slice held in one LDS stage
#ifndef RBMOE_STREAM_NW
#define RBMOE_STREAM_NW 4
#endif
constexpr int NW = RBMOE_STREAM_NW;     // waves per workgroup (4, or 8: one activation slice for twice the features)
constexpr int NT = NW * 64;
constexpr int CPR = BK / 8;            // 16-byte pieces per LDS row
constexpr int KS = BK / 16;            // matrix-core steps per slice
constexpr int TALL = 5;                // token blocks of a tall tile (see stream_tile_m; four otherwise)
constexpr int rows_of(int TT) { return 32 * TT; }                           // token rows per workgroup
constexpr int dma_per_wave(int TT) { return rows_of(TT) * CPR / 64 / NW; }  // LDS-DMA instructions per wave per slice
constexpr int RING = KS;    // weight-fragment steps in flight per wave (register ring depth)
constexpr int STAGES = 3;   // LDS stages of one activation slice each

// Token fragment read from LDS.
__device__ __forceinline__ bf16x8 lds_frag(const uint4* __restrict__ base, int idx) {
    return __builtin_bit_cast(bf16x8, base[idx]);
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// A pointer that is the same all over the wave, where the compiler does not see that it is.
__device__ __forceinline__ const char* scalar_pointer(const char* p) {
    const unsigned long long v = reinterpret_cast<unsigned long long>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)v), hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
    return reinterpret_cast<const char*>(((unsigned long long)hi << 32) | lo);
}

// Every vector-memory instruction of the main loop is issued from inline assembly and waited
// for by hand.  Left to the compiler, any wait that falls while an LDS-DMA is in flight
// becomes vmcnt(0), which drains the whole weight ring and the DMA just issued once per
// slice; and loads from read-only memory may be moved across the barriers the hand-written
// counts rely on.  Loads retire in order, so "at most N outstanding" proves that everything
// but the N youngest has landed; N is always the exact number of younger instructions.
__device__ __forceinline__ void issue_load(u32x4& d, uint32_t byte_off, const char* base) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(d) : "v"(byte_off), "s"(base));
}
__device__ __forceinline__ void issue_load(u32x2& d, uint32_t byte_off, const char* base) {
    asm volatile("global_load_dwordx2 %0, %1, %2" : "=v"(d) : "v"(byte_off), "s"(base));
}
// 64 lanes x 16 bytes from `src` (per lane) to LDS bytes [lds_addr, lds_addr + 1024).
__device__ __forceinline__ void issue_dma(uint32_t lds_addr, uint32_t byte_off, const char* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(byte_off), "s"(base) : "memory");
}
// Wait until at most N loads are outstanding; the two registers become usable only here.
template <int N, typename V>
__device__ __forceinline__ void wait_for(V& a, V& b) {
    asm volatile("s_waitcnt vmcnt(%2)" : "+v"(a), "+v"(b) : "n"(N));
}
template <int N>
__device__ __forceinline__ void wait_outstanding() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>), in order
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// f(0), f(1), ... while f returns true: slice I + 1 of a loop's remainder is reached only through slice I
template <int I, int N, typename F>
__device__ __forceinline__ void static_while(F&& f) {
    if constexpr (I < N) {
        if (f(std::integral_constant<int, I>{})) static_while<I + 1, N>(f);
    }
}

// One ring slot: the wave's two weight fragments of one reduction step.
// bf16: 16 bytes per lane per fragment, step g at byte 1024 g + 16 lane of a row block.
// int8: 8 bytes per lane per fragment; the packed layout is [K/32][64 lanes][16 bytes] with
//       bytes 0..7 for the even step and 8..15 for the odd one.
template <bool I8>
struct Slot;
template <>
struct Slot<false> {
    u32x4 f0, f1;
    __device__ __forceinline__ void load(const char* p0, const char* p1, int g, uint32_t lane16) {
        const uint32_t off = lane16 + (uint32_t)g * 1024u;
        issue_load(f0, off, p0);
        issue_load(f1, off, p1);
    }
    static __device__ __forceinline__ uint32_t offset(int g, uint32_t lane16) { return lane16 + (uint32_t)g * 1024u; }
    __device__ __forceinline__ void load0(const char* p0, uint32_t off) { issue_load(f0, off, p0); }
    __device__ __forceinline__ void load1(const char* p1, uint32_t off) { issue_load(f1, off, p1); }
    __device__ __forceinline__ bf16x8 a0() const { return __builtin_bit_cast(bf16x8, f0); }
    __device__ __forceinline__ bf16x8 a1() const { return __builtin_bit_cast(bf16x8, f1); }
};
template <>
struct Slot<true> {
    u32x2 f0, f1;
    __device__ __forceinline__ void load(const char* p0, const char* p1, int g, uint32_t lane16) {
        const uint32_t off = lane16 + (uint32_t)(g >> 1) * 1024u + (uint32_t)(g & 1) * 8u;
        issue_load(f0, off, p0);
        issue_load(f1, off, p1);
    }
    static __device__ __forceinline__ uint32_t offset(int g, uint32_t lane16) {
        return lane16 + (uint32_t)(g >> 1) * 1024u + (uint32_t)(g & 1) * 8u;
    }
    __device__ __forceinline__ void load0(const char* p0, uint32_t off) { issue_load(f0, off, p0); }
    __device__ __forceinline__ void load1(const char* p1, uint32_t off) { issue_load(f1, off, p1); }
    // pair i of the eight that the two fragments are, widened
    __device__ __forceinline__ uint32_t pair(int i) const {
        const u32x2& f = i < 4 ? f0 : f1;
        return widen2((i & 2) ? f.y : f.x, 16 * (i & 1));
    }
};

// ---- epilogue: the accumulators of one tile to memory -------------------------------------------------
struct TileOut {
    int rows, row0, tn_idx, N;
    bool act0, act1;      // whether the wave's two row blocks lie inside N
    int r0, r1;           // their first weight rows
    int t0, blocks;       // the wave's token blocks: the first of them, and how many
    int column;           // the wave's 32 features in the tile
    const float* sc;      // int8: the expert's scales, one per weight row
    bf16_t* out;
    bf16_t* gu_out;
    const bf16_t* bw_gu;
};

// `stage`: 256 bytes of LDS a row of the tile (32 KiB, tall tiles 40) that no wave of the workgroup reads or writes any more (the
// caller has made sure of that with a barrier).  `before_stores()` is called once, when the first pass has been converted and staged and
// before its first store to memory is issued.
template <bool SWIGLU, bool I8, int TT, bool HALVES, typename F>
__device__ __forceinline__ void write_tile(const TileOut& o, floatx16 (&acc)[2][TT], char* const stage,
                                           F&& before_stores) {
    constexpr int BN = SWIGLU ? NW * 32 : NW * 64, BM = rows_of(TT);
    // The thread index is made opaque here: everything derived from it below (LDS and row offsets, two dozen
    // values per lane) is then worked out where it is used.  Otherwise a caller that writes tile after tile has
    // them computed once, in front of its tile loop, and carried through the main loop in registers that the
    // loop does not have.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 31;
    const int lhalf = lane >> 5;
    const int rows = o.rows, row0 = o.row0, tn_idx = o.tn_idx, N = o.N, r0 = o.r0, r1 = o.r1;
    const bool act0 = o.act0, act1 = o.act1;
    const int column = HALVES ? o.column : wave;
    const int m0 = (HALVES ? o.t0 * 32 : 0) + lrow;  // the row of this lane's tokens in the wave's first block
    const float* const sc = o.sc;
    bf16_t* const out = o.out;
    bf16_t* const gu_out = o.gu_out;
    // Accumulator element v of block (b, t): feature 8*(v/4) + 4*(lane/32) + v%4 of the
    // wave's row block b, token t*32 + lane%32 - a lane holds 4 consecutive features of a
    // token, so a direct store would scatter 8-byte pieces over 32 rows per instruction.
    // Instead each block index goes through LDS as a tile of all its rows x 128 features (16-byte
    // pieces, piece p of row r kept at position p ^ (r % 16)), and is written out with
    // 16-byte stores, 16 consecutive lanes covering the 256 contiguous bytes of a row.
    // Passes through the staging tile: down product: the two blocks of 128 features; gate/up: the
    // hidden rows, then (only when the caller keeps them for a backward pass) the gate and the
    // up pre-activations, which go to `gu_out` [rows, 2N] with the gate half in columns [0, N).
    constexpr int PASSES = SWIGLU ? 3 : 2;
    constexpr int WH = NW < 4 ? NW : 4;  // waves that fill the staging tile at a time (32 features each)
    constexpr int SUB = NW / WH;         // ... in this many turns per block index
    constexpr int PW = WH * 4;           // 16-byte pieces of a staged row in use
#pragma unroll
    for (int bh = 0; bh < PASSES * SUB; ++bh) {
        const int b = bh / SUB, h = bh % SUB;
        if constexpr (SWIGLU) {
            // (uniform over the launch; a training layer's tiles are never tall)
            if (b > 0 && (TT >= TALL || gu_out == nullptr)) break;
        }
        if (bh) __syncthreads();  // the previous pass has been read out
        if ((wave / WH) == h && (SWIGLU ? act0 : (b ? act1 : act0))) {
            const int rb = b ? r1 : r0;
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                if (HALVES ? t >= o.blocks : t * 32 >= rows) continue;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int f = 8 * q + 4 * lhalf;  // first of 4 consecutive features inside the row block
                    float y[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (SWIGLU) {
                            float gv = acc[0][t][4 * q + i], uv = acc[1][t][4 * q + i];
                            if constexpr (I8) {
                                gv *= sc[r0 + f + i];
                                uv *= sc[r1 + f + i];
                            }
                            y[i] = b == 0 ? silu_bf16_grade(gv) * uv : (b == 1 ? gv : uv);
                        } else {
                            y[i] = acc[b][t][4 * q + i];
                            if constexpr (I8) y[i] *= sc[rb + f + i];
                        }
                    }
                    const int piece = ((column % WH) * 4 + q) ^ (lrow & 15);
                    *reinterpret_cast<uint2*>(stage + m0 * 256 + t * (32 * 256) + piece * 16 + lhalf * 8) =
                        make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
                }
            }
        }
        __syncthreads();
        if (bh == 0) before_stores();
        // where this pass goes: hidden rows and down rows into `out` (row stride N), the
        // pre-activations into `gu_out` (row stride 2 N)
        const int col0 = tn_idx * BN + (SWIGLU ? 0 : b * (NW * 32)) + h * (WH * 32);
        bf16_t* const dst = (SWIGLU && b > 0) ? gu_out + (b == 2 ? N : 0) : out;
        const size_t dstride = (SWIGLU && b > 0) ? (size_t)2 * N : (size_t)N;
#pragma unroll
        for (int i = 0; i < BM * PW / NT; ++i) {
            const int idx = i * NT + tid;
            const int r = idx / PW, p = idx % PW;
            if (r < rows && col0 + 8 * p < N) {
                const uint4 v = *reinterpret_cast<const uint4*>(stage + r * 256 + ((p ^ (r & 15)) * 16));
                uint4* const where = reinterpret_cast<uint4*>(dst + (size_t)(row0 + r) * dstride + col0 + 8 * p);
                if (SWIGLU && b > 0) {
                    // the pre-activations are not read again before the backward pass: stored past the caches,
                    // so that they do not push the hidden rows out before the down product reads them
                    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
                    __builtin_nontemporal_store(u32x4_t{v.x, v.y, v.z, v.w}, reinterpret_cast<u32x4_t*>(where));
                } else {
                    *where = v;
                }
            }
        }
    }
}

// The same for a launch whose product rows are the gradient of the hidden rows, SwiGlu::backward (src/ffn.rs:87-120)
// on the way out: with the gate and up pre-activations G | U of the forward pass, dG = dH * U * silu'(G) and
// dU = dH * silu(G) go to `gu_out` (both [rows, 2 N]) and the hidden gradient itself is never stored.  It passes through
// LDS in f32, 64 features at a time: rounded to bf16 first, as the tiles above are, it would cost the weight
// gradients a rounding more than the any-shape kernels' have (3.12e-3 from 64 bits against 2.81e-3).  A pass's
// pre-activations are requested in front of its barriers: 8192 tokens, d 768, 16 experts top-2 of 1408 take 80 us,
// 90 with the rounded tile and the requests behind them.
template <int TT>
__device__ __forceinline__ void write_swiglu_backward(const TileOut& o, floatx16 (&acc)[2][TT], char* const stage) {
    constexpr int BN = NW * 64;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 31, lhalf = lane >> 5;
    const int rows = o.rows, row0 = o.row0, N = o.N;
    constexpr int TURNS = rows_of(TT) * 8 / NT;
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int bh = 0; bh < NW; ++bh) {
        const int b = bh / (NW / 2), h = bh % (NW / 2);  // block index, pair of waves
        const int col0 = o.tn_idx * BN + b * (NW * 32) + h * 64;
        // this thread's pre-activations of the pass are under way while the tile is staged (read once: past the caches)
        u32x4_t g8[TURNS], u8[TURNS];
        auto offset_of = [&](int i, bool& in) {
            const int r = (i * NT + tid) / 8, p = tid % 8;  // 8 features of a row
            in = r < rows && col0 + 8 * p < N;
            return (size_t)(row0 + (in ? r : 0)) * 2 * N + (in ? col0 + 8 * p : 0);
        };
#pragma unroll
        for (int i = 0; i < TURNS; ++i) {
            bool in;
            const size_t off = offset_of(i, in);
            g8[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(o.bw_gu + off));
            u8[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(o.bw_gu + off + N));
        }
        if (bh) __syncthreads();  // the previous pass has been read out
        if (wave / 2 == h && (b ? o.act1 : o.act0)) {
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                if (t * 32 >= rows) continue;
                const int m = t * 32 + lrow;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<float4*>(stage + m * 256 + (((wave & 1) * 8 + 2 * q + lhalf) ^ (m & 15)) * 16) =
                        make_float4(acc[b][t][4 * q], acc[b][t][4 * q + 1], acc[b][t][4 * q + 2], acc[b][t][4 * q + 3]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TURNS; ++i) {
            bool in;
            const size_t off = offset_of(i, in);
            if (!in) continue;
            const int r = (i * NT + tid) / 8, p = tid % 8;
            const float4 lo = *reinterpret_cast<const float4*>(stage + r * 256 + ((2 * p) ^ (r & 15)) * 16);
            const float4 hi = *reinterpret_cast<const float4*>(stage + r * 256 + ((2 * p + 1) ^ (r & 15)) * 16);
            const float dh[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            const uint32_t gw[4] = {g8[i].x, g8[i].y, g8[i].z, g8[i].w}, uw[4] = {u8[i].x, u8[i].y, u8[i].z, u8[i].w};
            uint32_t dg[4], du[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float dgv[2], duv[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float gv = __uint_as_float(e ? gw[q] & 0xffff0000u : gw[q] << 16);
                    const float uv = __uint_as_float(e ? uw[q] & 0xffff0000u : uw[q] << 16);
                    const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gv * -1.44269504088896340736f));
                    dgv[e] = dh[2 * q + e] * uv * (sg * (1.0f + gv * (1.0f - sg)));  // silu', src/ffn.rs:235-238
                    duv[e] = dh[2 * q + e] * (gv * sg);
                }
                dg[q] = pack2(dgv[0], dgv[1]);
                du[q] = pack2(duv[0], duv[1]);
            }
            *reinterpret_cast<uint4*>(o.gu_out + off) = make_uint4(dg[0], dg[1], dg[2], dg[3]);
            *reinterpret_cast<uint4*>(o.gu_out + off + N) = make_uint4(du[0], du[1], du[2], du[3]);
        }
    }
}

// ---- the pipelined main loop: one memory instruction behind each multiply -------------------------
// A wave issues in order, and while it issues a vector-memory or LDS instruction it issues no multiply: with
// the loads of a step in one cluster in front of its eight multiplies the matrix core runs dry for the
// length of the cluster unless another wave of the SIMD fills in - a wave that is alone on its SIMD (the
// last round of a launch, the partner in its prologue or epilogue) reaches 64 % of the multiply rate that
// way.  Here every multiply is followed by at most one or two of them, in an order pinned by scheduling
// barriers, and the slice boundary has no cluster either: three LDS stages, and the workgroup barrier sits
// behind step KS - 2 of a slice, so that the last step of a slice can already read the first fragments of
// the next slice and issue the DMA of the slice after that into the stage the barrier has just proven free.
//   steps 0 .. KS-2 of slice k:  ring loads of step g + D, fragments of step g + 1 (stage k % 3)
//   then: wait for this wave's DMA of slice k + 1 (issued a slice ago), barrier
//   step KS-1:                   ring loads, DMA of slice k + 2 (into stage (k + 2) % 3, last read in
//                                slice k - 1), fragments of step 0 of slice k + 1 (stage (k + 1) % 3)
// Vector-memory issue order inside a step: ring f0, ring f1, then the DMA instructions.  Younger than the
// ring loads of step g when step g waits for them (they were issued in step g - D, D = 3): the DMA of that
// step if it was a last step, then two ring loads per step in between and four DMA if one of them was a last
// step - 8 in all for the steps 0 .. KS-2 of a slice, 4 for the last one.
// int8 weights are widened a step ahead, a pair or two behind each multiply: 24 instructions of eight cycles, which in front
// of the step's multiplies (256 cycles) left the matrix cores idle wherever the SIMD's other wave did not fill them.  So
// step g waits for the weights of step g + 1, and the loads of step g + 4 take the registers that step g's have left: issued
// in step g - 3 they have the same younger instructions.  A forward, d 768, 8 experts of 1408, widened in front / a step ahead:
// 3000 tokens 85.1 / 82.3 us, 4096 94.4 / 92.6, 8192 153.5 / 150.2 (gate/up at 4096 43.8 / 40.9 before the clock falls).
struct PipeCtx {
    const uint4* As;      // three LDS stages of one activation slice each
    uint32_t lds0;        // LDS byte address of this wave's rows in stage 0
    const char* a_base;   // activation rows (DMA source), byte offsets in a_src
    const char* wp0;      // this wave's two blocks of packed weight rows
    const char* wp1;
    uint32_t lane16;
    int lrow, lhalf, lxor;  // this lane's row in the wave's first token block
    int KT;               // slices of the reduction
};

// Before the call: the DMA of slices 0 and 1 (stages 0 and 1) and the ring loads of steps 0 .. D-1 have been issued
// and have landed, and the workgroup has met at a barrier.  After it: nothing is outstanding; every wave may
// still be reading the stages until the next barrier.
template <bool I8, int TT, int NB>
__device__ __forceinline__ void pipe_loop(const PipeCtx& c, floatx16 (&acc)[2][TT], Slot<I8> (&ring)[KS],
                                          const uint32_t (&a_src)[dma_per_wave(TT)]) {
    constexpr int D = I8 ? RING : RING - 1, BM = rows_of(TT), DMA_PER_WAVE = dma_per_wave(TT);
    static_assert(KS == 4 && RING == 4, "the wait counts below are derived for this configuration");
    const uint4* const As = c.As;
    const uint32_t lds0 = c.lds0, lane16 = c.lane16;
    const char* const a_base = c.a_base;
    const char* const wp0 = c.wp0;
    const char* const wp1 = c.wp1;
    const int lrow = c.lrow, lhalf = c.lhalf, lxor = c.lxor, KT = c.KT;
    const int GS = KT * KS;
    // The fragment of token block t for the step at position p of a slice sits at piece (2 p + lhalf) ^ lxor of
    // row t * 32 + lrow, i.e. at index t * 32 * CPR + (frag0 ^ 2 p): one register and an exclusive-or per step.
    // (Re-read through an empty statement per slice: four precomputed addresses would cost three registers.)
    static_assert(CPR == 8, "piece index = low three bits of the fragment index");
    int frag0 = lrow * CPR + (lhalf ^ lxor);
    bf16x8 tf[2][TT];
#pragma unroll
    for (int t = 0; t < NB; ++t) tf[0][t] = lds_frag(As, t * 32 * CPR + frag0);
    u32x4 wide[2][2];  // int8: the step's two fragments, and the next step's as they are widened
    if constexpr (I8)
        static_for<0, 8>([&](auto i) { wide[0][decltype(i)::value >> 2][decltype(i)::value & 3] = ring[0].pair(decltype(i)::value); });
    auto pslice = [&](int kt, auto idx_tag) {
        constexpr int IDX = decltype(idx_tag)::value;
        constexpr int BUF = IDX % 3, NEXT = (IDX + 1) % 3, FREE = (IDX + 2) % 3;
        const uint4* const Ab = As + BUF * (BM * CPR);
        const uint4* const An = As + NEXT * (BM * CPR);
        asm volatile("" : "+v"(frag0));
        static_for<0, KS>([&](auto s_tag) {
            constexpr int s = decltype(s_tag)::value;
            constexpr bool LAST = s == KS - 1;
            const int g = kt * KS + s;
            Slot<I8>& cur = ring[(I8 ? s + 1 : s) % RING];  // whose loads are awaited here
            Slot<I8>& nxt = ring[(s + D) % RING];
            wait_for<LAST ? 2 * (RING - 2) : 2 * (RING - 2) + DMA_PER_WAVE>(cur.f0, cur.f1);
            bf16x8 w0, w1;
            if constexpr (I8) {
                w0 = __builtin_bit_cast(bf16x8, wide[s & 1][0]);
                w1 = __builtin_bit_cast(bf16x8, wide[s & 1][1]);
            } else {
                w0 = cur.a0();
                w1 = cur.a1();
            }
            const uint32_t woff = Slot<I8>::offset(min(g + D, GS - 1), lane16);
            const uint32_t aoff = (uint32_t)min(kt + 2, KT - 1) * (BK * 2);
            const int frag = frag0 ^ (2 * ((s + 1) % KS));
            // memory instruction number i of the step
            constexpr int NOPS = 2 + ((LAST && DMA_PER_WAVE > NB) ? DMA_PER_WAVE : NB);
            auto op = [&](auto i_tag) {
                constexpr int i = decltype(i_tag)::value;
                if constexpr (i == 0) {
                    nxt.load0(wp0, woff);
                } else if constexpr (i == 1) {
                    nxt.load1(wp1, woff);
                } else {
                    constexpr int j = i - 2;
                    if constexpr (LAST && j < DMA_PER_WAVE)
                        issue_dma(lds0 + FREE * (BM * CPR * 16) + j * 8 * CPR * 16, a_src[j] + aoff, a_base);
                    if constexpr (j < NB)
                        tf[(s + 1) & 1][j] = lds_frag(LAST ? An : Ab, j * 32 * CPR + frag);
                }
            };
            static_for<0, 2 * NB>([&](auto m_tag) {
                constexpr int m = decltype(m_tag)::value;
                constexpr int b = m & 1, t = m >> 1;
                acc[b][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b ? w1 : w0, tf[s & 1][t], acc[b][t], 0, 0, 0);
                if constexpr (m < NOPS) op(m_tag);
                if constexpr (I8)
                    static_for<m * 8 / (2 * NB), (m + 1) * 8 / (2 * NB)>([&](auto i_tag) {
                        constexpr int i = decltype(i_tag)::value;
                        wide[(s + 1) & 1][i >> 2][i & 3] = cur.pair(i);
                    });
                __builtin_amdgcn_sched_barrier(0);
            });
            static_for<2 * NB, NOPS>(op);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (s == KS - 2) {
                // this wave's DMA of the next slice (issued in the last step of the slice before this
                // one) is older than the 2 * (KS - 1) ring loads of this slice so far
                wait_outstanding<2 * (KS - 1)>();
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };
    int kt = 0;
    for (; kt + 3 <= KT; kt += 3)
        static_for<0, 3>([&](auto i) { pslice(kt + decltype(i)::value, i); });
    static_while<0, 2>([&](auto i) {
        if (kt + decltype(i)::value >= KT) return false;
        pslice(kt + decltype(i)::value, i);
        return true;
    });
    wait_outstanding<0>();
    auto& ring_ref = ring;
#pragma unroll
    for (int i = 0; i < RING; ++i) asm volatile("" : : "v"(ring_ref[i].f0), "v"(ring_ref[i].f1));
}

// Which tile a workgroup takes.  Each XCD (workgroup number mod 8) walks a contiguous range of the launch's tiles, M
// fastest inside a group of row tiles; the tiles of the second, dense group (the shared expert's, in the same launch)
// come behind the routed ones, and its operands take the place of the routed experts' (all of it uniform over the
// workgroup).  `tm` < 0: no tile.
struct TileAt {
    int tm, tn;
    bool second;
};
template <int BN, int BM>
__device__ __forceinline__ TileAt tile_at(int tiles_m, int N, int group_m, int rows2, int N2) {
    int tiles_n = (N + BN - 1) / BN;
    const int total1 = tiles_m * tiles_n;
    const int tiles_n2 = (N2 + BN - 1) / BN, tiles_m2 = (rows2 + BM - 1) / BM;
    const int total = total1 + tiles_m2 * tiles_n2;
    const int per_xcd = (total + 7) / 8;
    const int local = blockIdx.x >> 3;
    int pid = (blockIdx.x & 7) * per_xcd + local;
    if (local >= per_xcd || pid >= total) return {-1, 0, false};
    const bool second = pid >= total1;
    if (second) {
        pid -= total1;
        tiles_n = tiles_n2;
        tiles_m = tiles_m2;
    }
    const int per_group = group_m * tiles_n;
    const int grp = pid / per_group;
    const int first_m = grp * group_m;
    const int gsize = min(group_m, tiles_m - first_m);
    const int in_g = pid - grp * per_group;
    return {first_m + in_g % gsize, in_g / gsize, second};
}

struct DenseGroup {
    const bf16_t* a;
    const void* w;
    const float* scales;
    int N, K, rows;
    bf16_t *out, *gu_out;
};

// OWN: the launch works its tiles out by itself (RoutedSlots); HALVES: its last feature tile may have at most 64 features.  Kernels
// of their own, since a workgroup's first loads wait for every instruction in front of them and the tables' code takes more scalar
// registers than there are (22 of them kept in vector registers in one kernel for all, none without it).  us a forward, one kernel for
// all / these: 8192 rows by 16 experts of 1408, d 768, 151.8 / 150.6; 2048 rows of the default model, which works its tiles out, 34.3 / 34.0
// (without the code for halves no faster: launches that work their tiles out always carry it).
template <bool SWIGLU, bool I8, int TT, bool OWN, bool HALVES>
__global__ __launch_bounds__(NT, RBMOE_STREAM_OCC) void grouped_stream_kernel(
    const bf16_t* __restrict__ a, const int* __restrict__ row_index, const void* __restrict__ wpacked,
    size_t w_expert_stride_bytes, const float* __restrict__ scales, size_t s_expert_stride, int N, int K,
    const int* __restrict__ tile_expert, const int* __restrict__ tile_row0, const int* __restrict__ tile_rows,
    const int* __restrict__ ntiles, int dense_rows, bf16_t* __restrict__ out, bf16_t* __restrict__ gu_out,
    const bf16_t* __restrict__ bw_gu, int group_m, DenseGroup g2, RoutedSlots slots) {
    constexpr int BN = SWIGLU ? NW * 32 : NW * 64;  // output features per workgroup
    constexpr int BM = rows_of(TT), DMA_PER_WAVE = dma_per_wave(TT);
    // LDS stages of one activation slice each; the epilogue reuses the first two as one
    // BM x 128 staging tile for the output.
    __shared__ uint4 As[STAGES * BM * CPR];

    // without tables: what the router left behind (RoutedSlots), worked out in the stages' room; the rows' tokens lie in the
    // stage that is filled last, behind a barrier
    static_assert(!OWN || (SWIGLU && TT < TALL), "");
    SlotsLds& sl = *reinterpret_cast<SlotsLds*>(As);
    static_assert(sizeof(SlotsLds) <= (STAGES - 1) * BM * CPR * sizeof(uint4), "in front of the tokens");
    int* const own_token = reinterpret_cast<int*>(As + (STAGES - 1) * BM * CPR);
    RoutedCounts rc{};
    if constexpr (OWN) {
        if (blockIdx.x == gridDim.x - 1) return routed_rest(slots, reinterpret_cast<unsigned char*>(As));
        rc = routed_counts<NT>(slots, sl);
    }
    const TileAt at = tile_at<BN, BM>(OWN ? rc.ntiles : dense_rows >= 0 ? (dense_rows + BM - 1) / BM : *ntiles, N, group_m, g2.rows, g2.N);
    if (at.tm < 0) return;
    const int tm_idx = at.tm, tn_idx = at.tn;
    if (at.second) {
        a = g2.a;
        row_index = nullptr;
        wpacked = g2.w;
        scales = g2.scales;
        N = g2.N;
        K = g2.K;
        dense_rows = g2.rows;
        out = g2.out;
        gu_out = g2.gu_out;
    }

    RBMOE_TRACE_AT(blockIdx.x, 0);
    int expert, row0, rows;
    if (dense_rows >= 0) {
        expert = 0;
        row0 = tm_idx * BM;
        rows = min(BM, dense_rows - row0);
    } else if constexpr (OWN) {
        const RoutedTile t = routed_tile<NT>(slots, rc, tm_idx, tn_idx == 0, sl, own_token);
        expert = t.expert;
        row0 = t.row0;
        rows = t.rows;
    } else {
        expert = tile_expert[tm_idx];
        row0 = tile_row0[tm_idx];
        rows = tile_rows[tm_idx];
    }
    const int nblk = (rows + 31) >> 5;  // token blocks that hold at least one row

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // ---- this wave's two blocks of 32 weight rows ---------------------------
    // A wave whose rows lie past N (ragged last feature tile) runs the same loop on row
    // block 0, so that every wave issues the same loads and meets the same barriers; it
    // stores nothing.
    // gate/up: gate rows nw .. nw + 31 and the matching up rows; down: rows nw .. nw + 31 and
    // the rows 128 further on, so that each block index covers 128 consecutive features of
    // the workgroup's tile.
    // A last gate/up tile of at most 64 features leaves two waves without any: there the waves share out the token blocks as well,
    // two blocks of features by two halves of the rows.  us a forward, without / with: 64 experts of 704 (five and a half tiles), six a
    // row, and a shared one of 1408, d 1024, 16384 rows 648 / 642; 32 of 704, int8, four a row, 8192 rows 205 / 200.
    static_assert(!HALVES || (SWIGLU && NW == 4), "");
    const bool halves = HALVES && nblk > 2 && N - tn_idx * BN <= 64;  // uniform over the workgroup
    const int column = halves ? wave & 1 : wave;
    // the wave's token blocks
    const int half = (nblk + 1) / 2, tb0 = halves ? (wave >> 1) * half : 0, tbs = halves ? min(half, nblk - tb0) : nblk;
    const int nw = tn_idx * BN + column * 32;
    const int r0 = nw, r1 = SWIGLU ? N + nw : nw + NW * 32;
    const bool act0 = nw < N;
    const bool act1 = SWIGLU ? act0 : (nw + NW * 32 < N);
    const size_t block_bytes = (size_t)K * 32 * (I8 ? 1 : 2);  // one block of 32 weight rows over all of K
    const char* wexp = static_cast<const char*>(wpacked) + (size_t)expert * w_expert_stride_bytes;
    const char* wp0 = wexp + (size_t)(act0 ? r0 / 32 : 0) * block_bytes;
    const char* wp1 = wexp + (size_t)(act1 ? r1 / 32 : 0) * block_bytes;
    if constexpr (OWN || HALVES || TT == TALL) {
        wp0 = scalar_pointer(wp0);
        wp1 = scalar_pointer(wp1);
    }
    const uint32_t lane16 = (uint32_t)lane * 16u;

    // ---- LDS-DMA of the activation slice --------------------------------------
    // Wave w fills a quarter of the LDS rows, from BM / NW * w on (32 rows, 40 of a tall tile): instruction j covers 8 of them,
    // lane l lands in row 8 j + l / 8 (of the wave's), position l % 8, and therefore
    // fetches logical piece (l % 8) ^ ((row / 2) % 8): a 16-lane group of a fragment read
    // (16 consecutive rows, one logical piece) then touches 8 distinct pieces in the even rows
    // and 8 in the odd rows, i.e. all 64 banks once.  Rows past the end of the group are
    // clamped to the tile's first row: their products are never stored.
    // Byte offsets from `a` fit 32 bits (the launcher checks rows * K * 2 < 4 GiB).
    const char* const a_base = reinterpret_cast<const char*>(a);
    uint32_t a_src[DMA_PER_WAVE];
#pragma unroll
    for (int j = 0; j < DMA_PER_WAVE; ++j) {
        const int r = wave * (BM / NW) + j * 8 + (lane >> 3);
        const int rr = r < rows ? r : 0;
        const int grow = OWN && !at.second ? own_token[rr] : row_index ? row_index[row0 + rr] : row0 + rr;
        a_src[j] = ((uint32_t)grow * (uint32_t)K + 8u * ((lane & 7) ^ ((r >> 1) & 7))) * 2u;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)As + wave * (BM / NW) * CPR * 16;
    auto dma_a = [&](int kt, auto buf_tag) {
        constexpr int BUF = decltype(buf_tag)::value;
#pragma unroll
        for (int j = 0; j < DMA_PER_WAVE; ++j)
            issue_dma(lds0 + BUF * (BM * CPR * 16) + j * 8 * CPR * 16, a_src[j] + (uint32_t)kt * (BK * 2), a_base);
    };

    floatx16 acc[2][TT];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[b][t][v] = 0.0f;

    const int lrow = lane & 31;
    const int lhalf = lane >> 5;
    const int lxor = (lrow >> 1) & 7;

    const int KT = K / BK;
    const int GS = KT * KS;  // reduction steps in all
    constexpr int D = I8 ? RING : RING - 1;  // the load for step g + D is issued while step g runs

    // ---- prologue: the first STAGES - 1 activation slices, the first D weight steps; nothing is in flight
    // where the loop is entered (the compiler may copy registers there)
    Slot<I8> ring[RING];
    static_for<0, STAGES - 1>([&](auto st) { dma_a(min((int)decltype(st)::value, KT - 1), st); });
#pragma unroll
    for (int g = 0; g < D; ++g) ring[g].load(wp0, wp1, min(g, GS - 1), lane16);
    wait_outstanding<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    RBMOE_TRACE_AT(blockIdx.x, 1);

    // The loop is specialised at compile time for the number of token blocks that hold rows: a run-time branch per
    // block between the multiplies costs far more than the skipped multiplies save.
    {
        const PipeCtx pc{As, lds0, a_base, wp0, wp1, lane16, tb0 * 32 + lrow, lhalf, lxor, KT};
        static_assert(TT >= 4 && TT <= 5, "one specialisation per possible block count");
        if (TT >= 5 && tbs >= 5) pipe_loop<I8, TT, (TT >= 5 ? 5 : TT)>(pc, acc, ring, a_src);
        else if (tbs >= 4) pipe_loop<I8, TT, 4>(pc, acc, ring, a_src);
        else if (tbs == 3) pipe_loop<I8, TT, 3>(pc, acc, ring, a_src);
        else if (tbs == 2) pipe_loop<I8, TT, 2>(pc, acc, ring, a_src);
        else pipe_loop<I8, TT, 1>(pc, acc, ring, a_src);
    }
    RBMOE_TRACE_AT(blockIdx.x, 2);
    // ---- epilogue -------------------------------------------------------------
    __syncthreads();  // every wave's last DMA has landed and its last fragment reads are done
    const TileOut to{rows, row0, tn_idx, N, act0, act1, r0, r1, tb0, tbs, column,
                     I8 ? scales + (size_t)expert * s_expert_stride : nullptr, out, gu_out, bw_gu};
    if constexpr (!SWIGLU && !I8 && TT < TALL) {
        if (bw_gu != nullptr) {  // uniform over the launch
            write_swiglu_backward<TT>(to, acc, reinterpret_cast<char*>(As));
            RBMOE_TRACE_AT(blockIdx.x, 3);
            return;
        }
    }
    write_tile<SWIGLU, I8, TT, HALVES>(to, acc, reinterpret_cast<char*>(As), [] {});
    RBMOE_TRACE_AT(blockIdx.x, 3);
}


// ---- the narrow kernel: launches with few tiles ------------------------------------------------------
// Half the weight rows a workgroup (a wave owns 128 token rows x ONE block of 32 weight rows) and a deep weight ring.
// With fewer workgroups than compute units the kernel above is bound by the latency of its weight loads: they run
// three steps (0.3 us) ahead, a first touch of expert weights takes one to two microseconds, and a lone workgroup took
// 1.1 us a slice of 64 columns whose multiplies last 0.43.  Half the accumulators leave registers for 16 steps of
// weights under way, a fourth LDS stage lets the DMA run three slices ahead, and there are twice as many workgroups.
// A full chip is better off with the kernel above: here each token fragment read from LDS serves one multiply instead
// of two.
//   gate/up: waves 0 and 1 take 64 gate rows, waves 2 and 3 the matching up rows, which meet in LDS at the end.
//   down:    four blocks of 32 features side by side.
// Issue order inside a step: the ring load, then (last step of a slice) the four DMA instructions.  Step g's ring load
// was issued in step g - 15; younger are 14 ring loads and the DMA of the last steps among g - 15 .. g - 1: four of
// them, three when g itself is one.  The DMA of slice kt + 1 was issued in the last step of slice kt - 2; when slice
// kt waits for it behind its step KS - 2, seven ring loads and the DMA of slice kt + 2 are younger.
constexpr int NRING = 16;
constexpr int NSTAGES = 4;
constexpr int TT = 4, BM = rows_of(TT), DMA_PER_WAVE = dma_per_wave(TT);  // (this kernel's tiles are never tall)
static_assert(BM == kStreamTileM, "");

template <bool I8>
struct Slot1;
template <>
struct Slot1<false> {
    u32x4 f;
    static __device__ __forceinline__ uint32_t offset(int g, uint32_t lane16) { return Slot<false>::offset(g, lane16); }
    __device__ __forceinline__ bf16x8 frag() const { return __builtin_bit_cast(bf16x8, f); }
};
template <>
struct Slot1<true> {
    u32x2 f;
    static __device__ __forceinline__ uint32_t offset(int g, uint32_t lane16) { return Slot<true>::offset(g, lane16); }
    __device__ __forceinline__ uint32_t pair(int i) const { return widen2((i & 2) ? f.y : f.x, 16 * (i & 1)); }
};

template <int N, typename V>
__device__ __forceinline__ void wait_for1(V& a) {
    asm volatile("s_waitcnt vmcnt(%1)" : "+v"(a) : "n"(N));
}

// As pipe_loop: before the call nothing is outstanding (slices 0 .. NSTAGES - 2 and ring steps 0 .. D - 1 have
// landed) and the workgroup has met at a barrier; after it nothing is outstanding.
template <bool I8, int NB>
__device__ __forceinline__ void narrow_loop(const PipeCtx& c, floatx16 (&acc)[TT], Slot1<I8> (&ring)[NRING],
                                            const uint32_t (&a_src)[DMA_PER_WAVE]) {
    constexpr int D = I8 ? NRING : NRING - 1;  // (int8 weights are widened a step ahead, as above)
    static_assert(KS == 4 && NRING == 16 && NSTAGES == 4 && DMA_PER_WAVE == 4 && TT == 4, "the wait counts are derived for this");
    const uint4* const As = c.As;
    const uint32_t lds0 = c.lds0, lane16 = c.lane16;
    const char* const a_base = c.a_base;
    const char* const wp = c.wp0;
    const int KT = c.KT, GS = KT * KS;
    int frag0 = c.lrow * CPR + (c.lhalf ^ c.lxor);
    bf16x8 tf[2][TT];
#pragma unroll
    for (int t = 0; t < NB; ++t) tf[0][t] = lds_frag(As, t * 32 * CPR + frag0);
    u32x4 wide[2];
    if constexpr (I8)
        static_for<0, 4>([&](auto i) { wide[0][decltype(i)::value] = ring[0].pair(decltype(i)::value); });
    auto pslice = [&](int kt, auto idx_tag) {
        constexpr int IDX = decltype(idx_tag)::value;  // kt % 4
        constexpr int NEXT = (IDX + 1) % NSTAGES, FREE = (IDX + 3) % NSTAGES;
        const uint4* const Ab = As + IDX * (BM * CPR);
        const uint4* const An = As + NEXT * (BM * CPR);
        asm volatile("" : "+v"(frag0));
        static_for<0, KS>([&](auto s_tag) {
            constexpr int s = decltype(s_tag)::value;
            constexpr bool LAST = s == KS - 1;
            constexpr int P = IDX * KS + s;  // ring position of step g
            const int g = kt * KS + s;
            Slot1<I8>& cur = ring[(I8 ? P + 1 : P) % NRING];  // whose load is awaited here
            wait_for1<(NRING - 2) + DMA_PER_WAVE * (LAST ? 3 : 4)>(cur.f);
            bf16x8 w;
            if constexpr (I8) w = __builtin_bit_cast(bf16x8, wide[s & 1]);
            else w = cur.frag();
            const uint32_t woff = Slot1<I8>::offset(min(g + D, GS - 1), lane16);
            const uint32_t aoff = (uint32_t)min(kt + 3, KT - 1) * (BK * 2);
            const int frag = frag0 ^ (2 * ((s + 1) % KS));
            constexpr int NOPS = 1 + (LAST ? DMA_PER_WAVE : NB);
            auto op = [&](auto i_tag) {
                constexpr int i = decltype(i_tag)::value;
                if constexpr (i == 0) {
                    issue_load(ring[(P + D) % NRING].f, woff, wp);
                } else {
                    constexpr int j = i - 1;
                    if constexpr (LAST)
                        issue_dma(lds0 + FREE * (BM * CPR * 16) + j * 8 * CPR * 16, a_src[j] + aoff, a_base);
                    if constexpr (j < NB) tf[(s + 1) & 1][j] = lds_frag(LAST ? An : Ab, j * 32 * CPR + frag);
                }
            };
            static_for<0, NB>([&](auto m_tag) {
                constexpr int m = decltype(m_tag)::value;
                acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, tf[s & 1][m], acc[m], 0, 0, 0);
                if constexpr (m < NOPS) op(m_tag);
                if constexpr (I8)
                    static_for<m * 4 / NB, (m + 1) * 4 / NB>([&](auto i_tag) {
                        constexpr int i = decltype(i_tag)::value;
                        wide[(s + 1) & 1][i] = cur.pair(i);
                    });
                __builtin_amdgcn_sched_barrier(0);
            });
            static_for<NB, NOPS>(op);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (s == KS - 2) {
                wait_outstanding<(2 * KS - 1) + DMA_PER_WAVE>();
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };
    int kt = 0;
    for (; kt + 4 <= KT; kt += 4)
        static_for<0, 4>([&](auto i) { pslice(kt + decltype(i)::value, i); });
    static_while<0, 3>([&](auto i) {
        if (kt + decltype(i)::value >= KT) return false;
        pslice(kt + decltype(i)::value, i);
        return true;
    });
    wait_outstanding<0>();
#pragma unroll
    for (int i = 0; i < NRING; ++i) asm volatile("" : : "v"(ring[i].f));
}

// PARTS: plain launches whose reduction is shared out (GroupedArgs::parts along y); kernels of their own, since the others' first loads
// wait for every instruction in front of them (203 rows by 16 experts, in whole, 46.4 us a block step, with one kernel for both 47.7).
template <bool SWIGLU, bool I8, bool PARTS>
__global__ __launch_bounds__(NT, 2) void narrow_grouped_stream_kernel(
    const bf16_t* __restrict__ a, const int* __restrict__ row_index, const void* __restrict__ wpacked,
    size_t w_expert_stride_bytes, const float* __restrict__ scales, size_t s_expert_stride, int N, int K,
    const int* __restrict__ tile_expert, const int* __restrict__ tile_row0, const int* __restrict__ tile_rows,
    const int* __restrict__ ntiles, int dense_rows, bf16_t* __restrict__ out, int group_m, DenseGroup g2, RoutedSlots slots,
    int part_rows) {
    constexpr int BN = SWIGLU ? 64 : 128;  // output features per workgroup
    __shared__ uint4 As[NSTAGES * BM * CPR];

    // without tables: what the router left behind (RoutedSlots), worked out in the stages' room; the rows' tokens lie in the
    // stage that is filled last, behind a barrier
    const bool own = SWIGLU && slots.expert_of != nullptr;  // uniform over the launch
    SlotsLds& sl = *reinterpret_cast<SlotsLds*>(As);
    static_assert(sizeof(SlotsLds) <= (NSTAGES - 1) * BM * CPR * sizeof(uint4), "in front of the tokens");
    int* const own_token = reinterpret_cast<int*>(As + (NSTAGES - 1) * BM * CPR);
    RoutedCounts rc{};
    if (own) {
        if (blockIdx.x == gridDim.x - 1) return routed_rest(slots, reinterpret_cast<unsigned char*>(As));
        rc = routed_counts<NT>(slots, sl);
    }
    const TileAt at = tile_at<BN, BM>(own ? rc.ntiles : dense_rows >= 0 ? (dense_rows + BM - 1) / BM : *ntiles, N, group_m, g2.rows, g2.N);
    if (at.tm < 0) return;
    const int tm_idx = at.tm, tn_idx = at.tn;
    if (at.second) {
        a = g2.a;
        row_index = nullptr;
        wpacked = g2.w;
        scales = g2.scales;
        N = g2.N;
        K = g2.K;
        dense_rows = g2.rows;
        if constexpr (PARTS) part_rows = g2.rows;
        out = g2.out;
    }
    const int n0 = tn_idx * BN;
    int expert, row0, rows;
    if (dense_rows >= 0) {
        expert = 0;
        row0 = tm_idx * BM;
        rows = min(BM, dense_rows - row0);
    } else if (own) {
        const RoutedTile t = routed_tile<NT>(slots, rc, tm_idx, tn_idx == 0, sl, own_token);
        expert = t.expert;
        row0 = t.row0;
        rows = t.rows;
    } else {
        expert = tile_expert[tm_idx];
        row0 = tile_row0[tm_idx];
        rows = tile_rows[tm_idx];
    }
    const int nblk = (rows + 31) >> 5;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // this wave's 32 weight rows; past N (ragged last feature tile) it runs the same loop on block 0 and stores nothing
    const int fb = n0 + (SWIGLU ? wave & 1 : wave) * 32;  // its first output feature
    const bool act = fb < N;
    const int wrow = SWIGLU && wave >= 2 ? N + fb : fb;
    const size_t block_bytes = (size_t)K * 32 * (I8 ? 1 : 2);
    int from = 0, KT = K / BK;  // this workgroup's slices of the reduction
    if constexpr (PARTS) {
        static_assert(!SWIGLU, "");
        const int parts = gridDim.y, to = KT * (blockIdx.y + 1) / parts;
        from = KT * blockIdx.y / parts;
        KT = to - from;
    }
    const int GS = KT * KS;
    const char* const wp = static_cast<const char*>(wpacked) + (size_t)expert * w_expert_stride_bytes +
                           (size_t)(act ? wrow / 32 : 0) * block_bytes + (size_t)from * BK * 32 * (I8 ? 1 : 2);
    const uint32_t lane16 = (uint32_t)lane * 16u;

    // LDS-DMA of the activation slices: as in the kernel above
    const char* const a_base = reinterpret_cast<const char*>(a);
    uint32_t a_src[DMA_PER_WAVE];
#pragma unroll
    for (int j = 0; j < DMA_PER_WAVE; ++j) {
        const int r = wave * (BM / NW) + j * 8 + (lane >> 3);
        const int rr = r < rows ? r : 0;
        const int grow = own && !at.second ? own_token[rr] : row_index ? row_index[row0 + rr] : row0 + rr;
        a_src[j] = ((uint32_t)grow * (uint32_t)K + (uint32_t)from * BK + 8u * ((lane & 7) ^ ((r >> 1) & 7))) * 2u;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)As + wave * (BM / NW) * CPR * 16;

    floatx16 acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;

    Slot1<I8> ring[NRING];
#pragma unroll
    for (int g = 0; g < (I8 ? NRING : NRING - 1); ++g) issue_load(ring[g].f, Slot1<I8>::offset(min(g, GS - 1), lane16), wp);
    static_for<0, NSTAGES - 1>([&](auto st) {
        constexpr int ST = decltype(st)::value;
#pragma unroll
        for (int j = 0; j < DMA_PER_WAVE; ++j)
            issue_dma(lds0 + ST * (BM * CPR * 16) + j * 8 * CPR * 16, a_src[j] + (uint32_t)min(ST, KT - 1) * (BK * 2), a_base);
    });
    wait_outstanding<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    {
        const int lrow = lane & 31;
        const PipeCtx pc{As, lds0, a_base, wp, nullptr, lane16, lrow, lane >> 5, (lrow >> 1) & 7, KT};
        if (nblk >= 4) narrow_loop<I8, 4>(pc, acc, ring, a_src);
        else if (nblk == 3) narrow_loop<I8, 3>(pc, acc, ring, a_src);
        else if (nblk == 2) narrow_loop<I8, 2>(pc, acc, ring, a_src);
        else narrow_loop<I8, 1>(pc, acc, ring, a_src);
    }
    __syncthreads();  // every wave's last DMA has landed and its last fragment reads are done

    // ---- epilogue: accumulator element v of lane l is feature 8 (v / 4) + 4 (l / 32) + v % 4, token t * 32 + l % 32
    char* const lds = reinterpret_cast<char*>(As);
    const int lrow = lane & 31, lhalf = lane >> 5;
    const float* const sc = I8 ? scales + (size_t)expert * s_expert_stride + (act ? wrow : 0) : nullptr;
    if constexpr (I8) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[t][v] *= sc[8 * (v >> 2) + 4 * lhalf + (v & 3)];
    }
    if constexpr (PARTS) {  // sums as they are
        float* const to = reinterpret_cast<float*>(out) + ((size_t)blockIdx.y * part_rows + row0) * N + fb + 4 * lhalf;
#pragma unroll
        for (int t = 0; t < TT; ++t)
            if (act && t * 32 + lrow < rows)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<float4*>(to + (size_t)(t * 32 + lrow) * N + 8 * q) =
                        make_float4(acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]);
        return;
    }
    constexpr int XCH = 2 * TT * 16 * 64 * 4;  // gate/up: the up waves' accumulators, 32 KiB; the output tile behind them
    char* const stage = lds + (SWIGLU ? XCH : 0);
    if constexpr (SWIGLU) {
        float4* const xch = reinterpret_cast<float4*>(lds) + (wave & 1) * (TT * 4 * 64) + lane;
        if (wave >= 2) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (t * 32 < rows)
                        xch[(t * 4 + q) * 64] =
                            make_float4(acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]);
        }
        __syncthreads();
        if (wave < 2) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (t * 32 < rows) {
                        const float4 u = xch[(t * 4 + q) * 64];
                        acc[t][4 * q + 0] = silu_bf16_grade(acc[t][4 * q + 0]) * u.x;
                        acc[t][4 * q + 1] = silu_bf16_grade(acc[t][4 * q + 1]) * u.y;
                        acc[t][4 * q + 2] = silu_bf16_grade(acc[t][4 * q + 2]) * u.z;
                        acc[t][4 * q + 3] = silu_bf16_grade(acc[t][4 * q + 3]) * u.w;
                    }
        }
    }
    // the output tile through LDS (16-byte pieces, piece p of row r at position p ^ (r % pieces)), then 16-byte stores
    constexpr int PW = BN / 8;
    if (act && (!SWIGLU || wave < 2)) {
        const int w = SWIGLU ? wave & 1 : wave;
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            if (t * 32 >= rows) continue;
            const int m = t * 32 + lrow;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<uint2*>(stage + m * (BN * 2) + ((w * 4 + q) ^ (m & (PW - 1))) * 16 + lhalf * 8) =
                    make_uint2(pack2(acc[t][4 * q], acc[t][4 * q + 1]), pack2(acc[t][4 * q + 2], acc[t][4 * q + 3]));
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < BM * PW / NT; ++i) {
        const int idx = i * NT + tid;
        const int r = idx / PW, p = idx % PW;
        if (r < rows && n0 + 8 * p < N)
            *reinterpret_cast<uint4*>(out + (size_t)(row0 + r) * N + n0 + 8 * p) =
                *reinterpret_cast<const uint4*>(stage + r * (BN * 2) + ((p ^ (r & (PW - 1))) * 16));
    }
}

// Up to how many wide tiles (as many as are likely, not the upper bound of the grid) the narrow kernel takes a launch.
// Down products, bf16, reductions over 512: as long as the narrow workgroups are about one a compute unit.  us a step, wide
// against narrow, d 768, K 1408: 48 tiles (203 rows over 16 experts) 17.2 / 10.6 (the launch alone), 117 tiles (2000 rows)
// 65.1 / 59.0, 129 (2500 rows over 8) 68.6 / 63.3, 141 (2500 rows over 16) 76.4 / 77.2, 165 (3000 rows) 78.8 / 79.8, 186 (3500)
// 90.7 / 95.1.  Short reductions (the default model's 384) are mostly first loads and stores: 156 tiles 47.5 / 46.2, 244
// tiles 69.4 / 67.4, 392 the same.  int8 weights: 129 tiles 65.6 / 66.0, 156 tiles 82.3 / 83.1, 180 tiles 83.9 / 84.2, 204 tiles
// 92.6 / 92.2; 156 tiles of 16 experts 78.8 / 79.7.
// Gate/up workgroups are twice as many per tile (64 features): 81 tiles (K 512) 39.9 / 38.9, 88 (int8, K 768) 43.9 / 41.7, 156
// 42.5 / 46.0, 176 (K 768, the launch alone) 15.0 / 16.5.
// Launches that keep or read pre-activations (training) stay with the wide kernel's epilogue.
constexpr int narrow_tiles(bool swiglu, int K) { return swiglu ? 128 : K <= 512 ? 250 : 140; }

// Tiles of a launch: `m` row tiles of the routed rows, `bm` rows each, and `bn` features.
int stream_tiles(const GroupedArgs& g, int m, int bm, int bn) {
    const GroupedArgs::Dense& d2 = g.dense2;
    return m * ((g.N + bn - 1) / bn) + (d2.rows + bm - 1) / bm * ((d2.N + bn - 1) / bn);
}
// Whether the narrow kernel takes a launch.
bool stream_narrow(const GroupedArgs& g) {
    if (g.gu_out || g.swiglu_grad_gu || (g.dense_rows < 0 && g.tile_m == rows_of(TALL))) return false;
    const int m = g.dense_rows >= 0 ? (g.dense_rows + BM - 1) / BM : g.likely_tiles > 0 ? g.likely_tiles : g.max_tiles;
    return stream_tiles(g, m, BM, g.swiglu ? NW * 32 : NW * 64) <= narrow_tiles(g.swiglu, g.K);
}

template <bool SWIGLU, bool I8>
hipError_t launch_t(const GroupedArgs& g, hipStream_t s) {
    constexpr int BN = SWIGLU ? NW * 32 : NW * 64;
    const GroupedArgs::Dense& d2 = g.dense2;
    const bool tall = g.dense_rows < 0 && g.tile_m == rows_of(TALL);
    const int bm = tall ? rows_of(TALL) : BM;
    const int tiles_m = g.dense_rows >= 0 ? (g.dense_rows + bm - 1) / bm : g.max_tiles;
    const int total = stream_tiles(g, tiles_m, bm, BN);
    if (total <= 0) return hipSuccess;
    const DenseGroup g2{static_cast<const bf16_t*>(d2.a), d2.w, d2.scales, d2.N, d2.K, d2.rows,
                        static_cast<bf16_t*>(d2.out), static_cast<bf16_t*>(d2.gu_out)};
    const int group_m = g.group_m > 0 ? g.group_m : 8;
    const int rest = SWIGLU && g.slots.expert_of ? 1 : 0;  // (routed_rest)
    const bool narrow = stream_narrow(g);
    if (g.parts != 1 && (!narrow || SWIGLU)) return hipErrorInvalidValue;
    if (narrow) {
        auto narrow_go = [&](auto parts) {
            RB_LAUNCH((narrow_grouped_stream_kernel<SWIGLU, I8, decltype(parts)::value>),
                      dim3((stream_tiles(g, tiles_m, BM, BN / 2) + 7) / 8 * 8 + rest, g.parts), dim3(NT), 0, s,
                      static_cast<const bf16_t*>(g.a), g.row_index, g.w, g.w_expert_stride * (I8 ? 1 : 2), g.scales,
                      g.s_expert_stride, g.N, g.K, g.tile_expert, g.tile_row0, g.tile_rows, g.ntiles, g.dense_rows,
                      static_cast<bf16_t*>(g.out), group_m, g2, g.slots, g.part_rows);
        };
        if (g.parts == 1) narrow_go(std::false_type{});
        else if constexpr (!SWIGLU) narrow_go(std::true_type{});
        return hipGetLastError();
    }
    auto launch = [&](auto tt, auto own, auto halves) {
        RB_LAUNCH((grouped_stream_kernel<SWIGLU, I8, decltype(tt)::value, decltype(own)::value, decltype(halves)::value>), dim3((total + 7) / 8 * 8 + rest), dim3(NT), 0, s,
                  static_cast<const bf16_t*>(g.a), g.row_index, g.w, g.w_expert_stride * (I8 ? 1 : 2), g.scales,
                  g.s_expert_stride, g.N, g.K, g.tile_expert, g.tile_row0, g.tile_rows, g.ntiles, g.dense_rows,
                  static_cast<bf16_t*>(g.out), static_cast<bf16_t*>(g.gu_out), static_cast<const bf16_t*>(g.swiglu_grad_gu),
                  group_m, g2, g.slots);
    };
    if (tall && rest) return hipErrorInvalidValue;
    const std::integral_constant<int, TT> whole{};
    if constexpr (SWIGLU) {
        auto half = [&](int n) { return (n + BN - 1) % BN < BN / 2; };  // (a last tile of at most half its features)
        const bool halves = NW == 4 && (half(g.N) || (d2.rows > 0 && half(d2.N)));
        constexpr std::bool_constant<NW == 4> some{};
        const std::integral_constant<int, TALL> high{};
        if (rest) launch(whole, std::true_type{}, some);
        else if (tall && halves) launch(high, std::false_type{}, some);
        else if (tall) launch(high, std::false_type{}, std::false_type{});
        else if (halves) launch(whole, std::false_type{}, some);
        else launch(whole, std::false_type{}, std::false_type{});
    } else if (tall) {
        launch(std::integral_constant<int, TALL>{}, std::false_type{}, std::false_type{});
    } else {
        launch(whole, std::false_type{}, std::false_type{});
    }
    return hipGetLastError();
}


}  // namespace

// Rows of the tiles of a call of so many routed rows: 128, or 160 (TALL).  A tall tile takes 1.19 times as long for 1.25 times the
// rows: a wave's weight fragments, which are two thirds of what passes a compute unit's L1 (32 KiB a slice of 64 columns for the four
// waves, beside 16 of rows), serve five multiplies instead of four, and there are fewer first loads and last stores.  Against that,
// launches end in whole tiles, and one table serves both products.  So the lengths are estimated - tiles a compute unit, 0.3 of the
// way to the next whole number, by the tile's reduction and 800 columns for its ends - and the tall tiles taken where they gain 2 %,
// above the sizes that the narrow kernel, a shared expert in the launch and gate/up launches that make the tables take.  How the rows
// fall on the experts is not known, and a last round more or less is 3 to 4 %: of 200 calls measured where the estimate speaks for
// them by 1 % (ten layers of 3000 to 16384 rows, bf16 and int8, rows evenly spread and 30 % of them to one expert) they are 1.5 %
// faster on average and 19 slower by more than 1.5 %, of the 164 with 2 % 1.9 % faster and 8 slower, by 4 % at most.  Not for calls
// with padding, whose rows are fewer than the host knows: 30 of 100 with 30 % of it slower by more than 1.5 %, 0.2 % faster on
// average.  us a forward, 128 / 160, measured (estimated gain): d 768, 8 experts of 1408, 6000
// rows 113.2 / 108.1 (8 %), 10000 155.7 / 157.6 (1 %, not taken), 16384 235.3 / 224.2 (7 %); 16 of them, 6000 121.2 / 112.7 (8 %),
// 16384 251.4 / 246.1 (4 %); d 512, 8 of 352, 16384 90.5 / 83.4 (9 %); d 1024, 32 of 1408, four a row, 6000 256.6 / 244.8 (2 %),
// 16384 592 / 567 (4 %); 64 of 704, six a row, 16384 522 / 508 (3 %); d 256, 32 of 704, four a row, 10000 104.1 /
// 104.7 (3 %), 16384 143.9 / 135.9 (5 %).  Slower all the same: d 1024, 16 of 704, four a row, 8400 246 /
// 253.  Not taken: d 1024, 32 of 352, four a row, 10000 164.9 / 167.3, d 512, 8 of 1408, 6000 88.9 / 89.6, d 768, 8 of 1408, 8400 149.5 / 154.8,
// d 1024, 16 of 704, four a row, 5300 176.7 / 180.5, 64 of 704, six a row, 6000 237.7 / 231.0.
int stream_tile_m(int rows, int groups, int F, int d) {
    auto tiles = [&](int bm) { return std::max((double)rows / bm + 0.5 * groups, (double)std::min(groups, rows)); };
    const int gate_up = (F + 127) / 128, down = (d + 255) / 256;
    if (tiles(BM) * gate_up <= 768) return BM;
    auto length = [&](int bm) {
        auto units = [&](double n) { return n <= 256 ? 1.0 : 0.3 * std::ceil(n / 256) + 0.7 * n / 256; };
        return (d + 800) * units(tiles(bm) * gate_up) + (F + 800) * units(tiles(bm) * down);
    };
    return length(BM) > 1.02 * 1.19 * length(rows_of(TALL)) ? rows_of(TALL) : BM;
}

// A narrow down launch of few tiles waits for a chain of slices that holds a fraction of the compute units.  Its reduction is shared out
// where it is long and the rows, which the combine then reads in f32 and twice or four times, are few.  us a forward, whole / 2 parts
// / 4 parts (tiles; rows times d in thousands): d 512, 8 experts of 1408, 100 rows (32; 102) 31.5 / 29.9 / 30.1, 400 rows (40; 410) 35.4 /
// 34.2 / 34.3, 700 rows (56; 717) 36.2 / 36.4 / 36.5; d 768, 8 of 1408, int8, 83 rows (48; 127) 34.9 / 32.7 / 31.4, 200 rows (48; 307) 35.8 /
// 34.5 / 35.2; with a shared expert, bf16, 83 rows (54; 191) 36.1 / 35.7 / 36.5, 340 rows (72; 783) 40.7 / 41.3 / 41.3; 16 of 1408, 203 rows
// (96; 312) 40.6 / 41.2 / 41.1; d 1024, 8 of 1408, int8, 150 rows (64; 307) 37.7 / 36.0 / 37.8; 4 of 2730, 100 rows (32; 102) 39.7 / 35.7 / 35.0.
// Reductions of 384 and 704 lose: d 512, 8 of 352 and a shared one, 100 rows 26.0 / 26.9 / 26.7.  Over 560 shapes (d 256 to 1024, 4 to 16
// experts of 1024 to 2752, one to four a row, 40 to 640 rows) the rule gives 3.9 % a forward on average; 43 of them, of 1088 and, in bf16, 1408
// columns, are slower by 1.5 to 4.9 %: d 768, 4 of 1088, four a row, 64 rows 33.4 / 35.1 / 36.3, 8 of 1408 and a shared one, 186 rows
// 35.6 / 36.2 / 36.8.  (Lines drawn by the estimated gain leave out all but 4 of those and give 4.2 %, but round the rows of a call in other
// places than before: the lines stay.)
int stream_parts(const GroupedArgs& g) {
    if (g.swiglu || g.dense_rows >= 0 || !stream_narrow(g)) return 1;
    const int m = g.likely_tiles > 0 ? g.likely_tiles : g.max_tiles, tiles = stream_tiles(g, m, BM, 128);
    const int K = g.dense2.rows > 0 ? std::min(g.K, g.dense2.K) : g.K;
    const long long elements = (long long)(g.routed_rows + g.dense2.rows) * g.N;
    if (K < 1024 || tiles > 64 || elements > 512 * 1024) return 1;
    return tiles <= 48 && elements <= 128 * 1024 ? 4 : 2;
}

// K a multiple of 64 (one LDS slice), N a multiple of 32 (row blocks of the packed weights)
bool stream_shape_ok(int N, int K) { return K % 64 == 0 && K >= 64 && N % 32 == 0 && N >= 32; }

hipError_t launch_grouped_stream(const GroupedArgs& g, WeightKind wk, hipStream_t s) {
    if (!stream_shape_ok(g.N, g.K)) return hipErrorInvalidValue;
    if (g.dense2.rows > 0 && (!stream_shape_ok(g.dense2.N, g.dense2.K) || !g.dense2.gu_out != !g.gu_out || g.swiglu_grad_gu))
        return hipErrorInvalidValue;
    if (g.slots.expert_of && (!g.swiglu || g.dense_rows >= 0 || g.slots.layout.tile_m != BM)) return hipErrorInvalidValue;
    if (g.dense_rows < 0 && g.tile_m != BM && g.tile_m != rows_of(TALL)) return hipErrorInvalidValue;
    if (g.dense_rows < 0 && g.tile_m == rows_of(TALL) && (g.gu_out || g.swiglu_grad_gu)) return hipErrorInvalidValue;
    if (g.swiglu_grad_gu && (g.swiglu || wk != WeightKind::BF16)) return hipErrorInvalidValue;
    if (wk == WeightKind::BF16) return g.swiglu ? launch_t<true, false>(g, s) : launch_t<false, false>(g, s);
    if (wk == WeightKind::I8) return g.swiglu ? launch_t<true, true>(g, s) : launch_t<false, true>(g, s);
    return hipErrorInvalidValue;
}

// Host-side repacking of one [rows, cols] weight matrix into fragment order.
// bf16: [rows/32][cols/16][64 lanes][8]; lane l holds row (l % 32), columns 16*s + 8*(l/32) + 0..7.
void pack_weight_bf16(const uint16_t* src, int rows, int cols, uint16_t* dst) {
    const int KS16 = cols / 16;
    for (int nb = 0; nb < rows / 32; ++nb)
        for (int s = 0; s < KS16; ++s)
            for (int l = 0; l < 64; ++l) {
                const uint16_t* p = src + (size_t)(nb * 32 + l % 32) * cols + 16 * s + 8 * (l / 32);
                uint16_t* q = dst + (((size_t)nb * KS16 + s) * 64 + l) * 8;
                for (int j = 0; j < 8; ++j) q[j] = p[j];
            }
}

// int8: [rows/32][cols/32][64 lanes][16]; bytes 0..7 are the lane's piece of step 2s, bytes 8..15 of step 2s+1.
void pack_weight_i8(const int8_t* src, int rows, int cols, int8_t* dst) {
    const int KS32 = cols / 32;
    for (int nb = 0; nb < rows / 32; ++nb)
        for (int s = 0; s < KS32; ++s)
            for (int l = 0; l < 64; ++l) {
                const int8_t* p = src + (size_t)(nb * 32 + l % 32) * cols + 32 * s + 8 * (l / 32);
                int8_t* q = dst + (((size_t)nb * KS32 + s) * 64 + l) * 16;
                for (int j = 0; j < 8; ++j) {
                    q[j] = p[j];
                    q[8 + j] = p[16 + j];
                }
            }
}

}  // namespace rbmoe
