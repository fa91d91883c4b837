// Routing code shared by the large-batch and the decode-shaped kernels: norm, logits, softmax and top-k of a block of
// tokens whose rows lie in LDS as a whole.
#pragma once

#include "rbmoe_kernels.h"

namespace rbmoe {

// Dynamic LDS layout of router_kernel (floats / ints, in this order):
//   prob   [TB][ES]   logits, then exp, then probabilities   (ES = E | 1)
//   lsev   [TB]       log-sum-exp per token
//   gates  [TB][k]    selected probabilities, then gates
//   lexp   [TB][k]    selected expert per local slot (-1 = unrouted)
//   wcount [waves][E] per-wave match counts of one ranking round
//   running[E]        slots already ranked per expert
__host__ __device__ static size_t router_fixed_bytes(int E, int k, int tokens = kRouterTokens) {
    const int ES = E | 1;
    size_t n = (size_t)tokens * ES + tokens + 2 * (size_t)tokens * k + (size_t)kRouterWaves * E + E;
    return (n * 4 + 15) & ~(size_t)15;
}

// softmax, log-sum-exp and the k argmax rounds for the tokens of one wave of a router block (see router_tail).
// Everything order-sensitive keeps the reference's order: the maximum ignores NaN (f32::max), exp(v - max) is
// summed one expert after the other in index order, the k argmax rounds prefer the lower index on equal
// probabilities, and the gates are summed in rank order.
// The sum: lane l of a group holds ((ex_0 + ex_1) + ... ) + ex_l after l steps of "take the lane below's sum,
// add your own value" (a shift of the whole wave by one lane inside the add; a group's first lane starts from the sum
// carried over from the experts of the slices before) - the reference's chain, one rounded add per expert, with
// no trip through LDS; lanes past the last expert add zeros.  What a group's first lane takes in from the group below
// follows one lane behind and is overtaken by nobody: the last lane's sum after G - 1 steps is the chain's.  An argmax round is two reductions of 32 bits: the
// greatest probability bits (probabilities are never negative, so the bits order like the values), then the
// lowest expert index among the lanes that hold them.
// NQ = turns a wave needs for its tokens (64 / G tokens a turn); the NQ turns share no data and run interleaved.
template <int MAXJ, int NQ, int TB>
__device__ __forceinline__ void softmax_topk(float* __restrict__ prob, float* __restrict__ lsev,
                                             float* __restrict__ gates, int* __restrict__ lexp, int G, int t0, int nt,
                                             int ES, const uint8_t* __restrict__ valid, int E, int k) {
    constexpr int TW = TB < kRouterWaves ? 1 : TB / kRouterWaves;  // tokens of a wave
    const int lane_ = threadIdx.x & 63, wave_ = threadIdx.x >> 6;
    const int lig = lane_ & (G - 1);          // lane in group
    const int gbase = lane_ & ~(G - 1);       // first lane of the group
    const int tpw = 64 / G;                   // tokens a wave handles in one turn
    const unsigned long long gmask = (G == 64 ? ~0ull : ((1ull << G) - 1ull)) << gbase;
    const float neg_inf = __uint_as_float(0xff800000u);
    int tok[NQ];
    bool live[NQ], ok[NQ];
    float* row[NQ];
    float pv[NQ][MAXJ], mx[NQ], sum[NQ], total[NQ];
    unsigned taken_bits[NQ];  // bit j: expert lig + G j is taken
    uint8_t in_use[NQ];       // (asked for here, looked at behind the softmax)
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        tok[q] = wave_ * TW + q * tpw + lane_ / G;  // token of this group in turn q
        live[q] = tok[q] < nt && tok[q] < (wave_ + 1) * TW && q * tpw < TW;
        in_use[q] = valid != nullptr ? valid[t0 + (live[q] ? tok[q] : 0)] : 1;
        row[q] = prob + (live[q] ? tok[q] : 0) * ES;
        mx[q] = neg_inf;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int e = lig + G * j;
            pv[q][j] = (live[q] && e < E) ? row[q][e] : neg_inf;
            const float vv = (pv[q][j] == pv[q][j]) ? pv[q][j] : neg_inf;  // a NaN never becomes the maximum
            mx[q] = vv > mx[q] ? vv : mx[q];
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) mx[q] = group_fmax(mx[q], G);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int e = lig + G * j;
            // lanes without an expert carry +0 through the sums below
            pv[q][j] = (live[q] && e < E) ? rb_expf(__fadd_rn(pv[q][j], -mx[q])) : 0.0f;
        }
    }
    // the sums: one chain of adds per token in index order, slice after slice
    {
        float carry[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) carry[q] = 0.0f;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            if (G * j >= E) break;  // uniform
            float acc[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) acc[q] = __fadd_rn(carry[q], pv[q][j]);  // in a group's first lane: 0 + ex_0 = ex_0 in the first slice
            for (int st = 1; st < G; ++st) {
#pragma unroll
                for (int q = 0; q < NQ; ++q)
                    acc[q] = __fadd_rn(__uint_as_float(lanes_from<0x138>(__float_as_uint(acc[q]))), pv[q][j]);  // wave_shr:1
            }
#pragma unroll
            for (int q = 0; q < NQ; ++q) carry[q] = __shfl(acc[q], gbase + G - 1);
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) sum[q] = carry[q];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        if (live[q] && lig == 0) lsev[tok[q]] = __fadd_rn(mx[q], rb_logf(sum[q]));
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int e = lig + G * j;
            if (live[q] && e < E) {
                if (sum[q] > 0.0f) pv[q][j] = __fdiv_rn(pv[q][j], sum[q]);
                row[q][e] = pv[q][j];
            }
        }
        ok[q] = live[q] && in_use[q] != 0;
        taken_bits[q] = 0;
        total[q] = 0.0f;
    }
    // ---- k rounds of argmax over the experts not yet taken ----
    // Without a NaN anywhere in the wave (with one expert a lane): the greatest probability bits among the untaken, then the
    // lowest of the lanes that hold them.
    bool any_nan = false;
#pragma unroll
    for (int q = 0; q < NQ; ++q) any_nan = any_nan || pv[q][0] != pv[q][0];
    if (MAXJ == 1 && __ballot(any_nan) == 0ull) {  // uniform over the wave
        bool open[NQ];  // this lane has an expert and it is not taken
#pragma unroll
        for (int q = 0; q < NQ; ++q) open[q] = live[q] && lig < E;
        for (int r = 0; r < k; ++r) {
            uint32_t best[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) best[q] = group_umax(open[q] ? __float_as_uint(pv[q][0]) : 0u, G);
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const unsigned long long holders = __ballot(open[q] && __float_as_uint(pv[q][0]) == best[q]) & gmask;
                const bool mine = holders != 0ull && (holders & ((1ull << lane_) - 1ull)) == 0ull && ((holders >> lane_) & 1ull);
                open[q] = open[q] && !mine;
                total[q] = __fadd_rn(total[q], __uint_as_float(best[q]));
                if (mine) {
                    lexp[tok[q] * k + r] = ok[q] ? lig : -1;
                    gates[tok[q] * k + r] = ok[q] ? __uint_as_float(best[q]) : 0.0f;
                }
            }
        }
    } else
    for (int r = 0; r < k; ++r) {
        int first[NQ];
        uint32_t lbits[NQ], le[NQ];  // this lane's best candidate: probability bits and expert index
        bool has[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            // First expert not yet taken: the lowest set bit of a ballot over the group, taking
            // the expert slices j in increasing order (slice j holds experts G j .. G j + G - 1).
            first[q] = 0x7fffffff;
#pragma unroll
            for (int j = MAXJ - 1; j >= 0; --j) {
                const int e = lig + G * j;
                const unsigned long long m = __ballot(e < E && !((taken_bits[q] >> j) & 1u)) & gmask;
                if (m != 0ull) first[q] = (__ffsll((long long)m) - 1 - gbase) + G * j;
            }
            // best candidate of this lane: not taken, not NaN; greater probability, then lower index
            has[q] = false;
            lbits[q] = 0;
            le[q] = 0x7fffffffu;
#pragma unroll
            for (int j = 0; j < MAXJ; ++j) {
                const int e = lig + G * j;
                if (live[q] && e < E && !((taken_bits[q] >> j) & 1u) && pv[q][j] == pv[q][j]) {
                    const uint32_t bits = __float_as_uint(pv[q][j]);
                    if (!has[q] || bits > lbits[q]) {  // slices in increasing index order: a tie keeps the lower index
                        lbits[q] = bits;
                        le[q] = (uint32_t)e;
                    }
                    has[q] = true;
                }
            }
        }
        uint32_t mbits[NQ], ci[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) mbits[q] = group_umax(has[q] ? lbits[q] : 0u, G);
#pragma unroll
        for (int q = 0; q < NQ; ++q) ci[q] = group_umin((has[q] && lbits[q] == mbits[q]) ? le[q] : 0x7fffffffu, G);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            // the reference starts from the first untaken expert and replaces it only on a
            // strictly greater probability: if that first one is NaN nothing replaces it
            bool first_nan = false;
#pragma unroll
            for (int j = 0; j < MAXJ; ++j)
                if (lig + G * j == first[q] && pv[q][j] != pv[q][j]) first_nan = true;
            const bool nan_wins = (__ballot(first_nan) & gmask) != 0ull;
            const bool use_first = nan_wins || ci[q] == 0x7fffffffu;
            const int best = use_first ? first[q] : (int)ci[q];
            float mine = 0.0f;
#pragma unroll
            for (int j = 0; j < MAXJ; ++j)
                if (lig + G * j == best) {
                    mine = pv[q][j];
                    taken_bits[q] |= 1u << j;
                }
            // the winner's probability is the greatest bits themselves; only a NaN first expert has to be fetched
            float bestv = __uint_as_float(mbits[q]);
            if (__ballot(use_first) != 0ull) {  // uniform over the wave
                const float fv = __shfl(mine, gbase + (best & (G - 1)));
                if (use_first) bestv = fv;
            }
            total[q] = __fadd_rn(total[q], bestv);
            if (live[q] && lig == 0) {
                lexp[tok[q] * k + r] = ok[q] ? best : -1;
                gates[tok[q] * k + r] = ok[q] ? bestv : 0.0f;
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        if (ok[q] && total[q] > 0.0f)
            for (int r = lig; r < k; r += G) gates[tok[q] * k + r] = __fdiv_rn(gates[tok[q] * k + r], total[q]);
}

// ---------------------------------------------------------------------------
// route_rows_body: norm (optional), logits and everything behind them for TB = 8, 16 or 32 tokens a workgroup, with
// the workgroup's whole rows in LDS at once.
// What bounds routing up to some thousand tokens is not work but the length of one workgroup's chain: with 32 tokens a
// workgroup and slices of columns staged in turn (route_fused_kernel) it takes 18 to 20 us whether 7 workgroups run or
// 256.  So the tokens of a workgroup are chosen to spread the call over the chip, everything a workgroup reads is
// requested in one batch, and a dot product is taken by NL neighbouring threads, thread j owning column lane j of the
// reference's sum: a chain of d / NL rounded multiplies and adds.  A thread works on TT tokens x EE experts side by
// side, so that TT + EE words read from LDS feed TT * EE products; its columns j, j + NL, ... lie side by side in LDS,
// so that it reads four steps of the chain at a time.
// NL = 8: `dot` (src/matrix.rs:26-40).  NL = 32: the quantized router's dot_lanes::<32> (src/quantized.rs:154-177), its
// int8 rows widened on their way into LDS, the sum times the row's scale (:61).
// The norm is RmsNorm::forward (src/norm.rs:41-61), its squares added up in index order as the reference does: a wave a row
// (ordered_sum_wave) straight from memory, which lays the normed row down - or, at widths that do not divide among its lanes,
// squares in column order beside the rows and one thread a row.
// Measured, against route_fused_kernel (and the norm's launch in front of it): d 768, 203 tokens x 16 experts 9.5 us
// against 18.1, with the norm 11.2 (one chain a row 14.4) against 32.2; 4096 x 8 10.1 against 17.7; 8192 x 16 17.3 against
// 19.0 (median inside a forward 20.9 against 22.8).  With the norm, 8 tokens of d 768 by a quantized router of 8 experts:
// rows there 1.2 us into the workgroup, their sums at 2.6, normed rows at 3.1, router rows in place at 3.7, logits at 6.9,
// softmax and top-k at 9.1, end 9.4.
// ---------------------------------------------------------------------------
struct RouteRowsArgs {
    const void* x;
    const float* wr;
    const int8_t* wq;
    const float* wscale;
    const float* bias;
    const uint8_t* valid;
    int T, d, E, k, EG;  // EG: experts whose router rows are in LDS together
    float* P;
    float* lse;
    int* expert_of;
    float* gate_of;
    int* rank_in_block;
    int* blockcnt;
    float* partial;
    bf16_t* rows16;
    const float* norm_w;
    float norm_eps;
    void* xn_out;
    int slice = 0;          // route_rows_kernel: experts of a workgroup (0: all of them)
    int* arrive = nullptr;  // ... and, with a slice, a token block's arrival counter, kDecodeCombineCounterStride apart
};
// A staged row: column lane j's elements side by side, `lane_pitch` floats from one lane to the next - whole 16-byte
// pieces (a last one short of four steps is filled up with zeros, which the sums do not see), and an odd number of
// them, so that the lanes' pieces start in different banks.
__host__ __device__ static int route_lane_pitch(int d, int NL) {
    const int steps = (d / NL + 3) / 4;
    return 4 * (steps | 1);
}
// Floats of the room that the router's rows and - before them - the squares share.
__host__ __device__ static int route_shared_floats(int d, int TB, int EG, int pitch, bool norm) {
    const int router = EG * pitch, squares = norm ? TB * (d + 4) + 64 : 0;  // (64: the chain reads ahead)
    return router > squares ? router : squares;
}
__host__ __device__ static size_t route_rows_lds_bytes(int E, int k, int d, int TB, int NL, int EG, bool norm) {
    const int pitch = NL * route_lane_pitch(d, NL);
    const bool chain = norm && !wave_norms(d);
    return router_fixed_bytes(E, k, TB) +
           ((size_t)TB * pitch + route_shared_floats(d, TB, EG, pitch, chain) + (chain ? d + TB : 0)) * 4;
}

// The logits of the TB tokens of block `blk` for the experts [e_from, e_to) into the `prob` array (row pitch E | 1) of `lds_raw`, with everything in
// front of them; the caller meets at a barrier before it reads them.  Kernels without the norm are compiled without its code:
// with it (a wave's row at four widths, a thread's at any) they are 90 to 126 KB long instead of 35 to 63 and take 139 to 152
// registers instead of 71 to 92, and 4096 tokens of d 768 by 8 experts are routed in 10.4 us instead of 10.1.  Both hold the
// body twice, with all experts and with some; a launch runs one of them.  From swept caches, where code is fetched too, 203
// tokens of d 768 by 16 experts are routed in 10.1 us, by the kernels of 26 KB with everything in one body in 10.8.
template <typename XT, int TB, int NL, int TT, int EE, bool NORM>
__device__ __forceinline__ void route_rows_body(const RouteRowsArgs& a, int blk, int e_from, int e_to,
                                                unsigned char* __restrict__ lds_raw) {
    constexpr int NT = kRouterThreads;
    const int T = a.T, d = a.d, E = a.E, k = a.k, EG = a.EG;
    const int ES = E | 1;
    constexpr bool norm = NORM;
    const bool wave_norm = norm && wave_norms(d);
    float* const prob = reinterpret_cast<float*>(lds_raw);
    const int lp = route_lane_pitch(d, NL), pitch = NL * lp;
    float* const xs = reinterpret_cast<float*>(lds_raw + router_fixed_bytes(E, k, TB));
    float* const ws = xs + TB * pitch;
    // with a norm: the rows' squares, d + 4 floats apart (their chains read from different banks), in the place of the
    // router's rows, which are put there behind the chains; the norm's weights and the rows' factors
    float* const sq = ws;
    const int sp = d + 4;
    float* const nws = ws + route_shared_floats(d, TB, EG, pitch, norm);
    float* const inv = nws + d;
    const int tid = threadIdx.x;
    const int t0 = blk * TB;
    const int nt = min(TB, T - t0);

    // Staging: 16-byte pieces of the router's rows and of the token rows, six of each a thread requested before the first
    // is stored (96 KB a trip to memory; variables of their own: an array of them ends up in scratch memory).  A row's
    // pieces are counted by a rounded-up reciprocal, exact for the few thousand there are.
    constexpr int XN = Vec16<XT>::N;
    const int wpr = NL == 32 ? d / 16 : d / 4, xpr = d / XN;
    const uint32_t wrecip = (uint32_t)(0x100000000ull / (uint32_t)wpr) + 1u, xrecip = (uint32_t)(0x100000000ull / (uint32_t)xpr) + 1u;
    auto put_router = [&](int i, const uint4& v) {
        const int r = wpr == 1 ? i : (int)__umulhi((uint32_t)i, wrecip), c = i - r * wpr;
        if constexpr (NL == 32) {
            float* const to = ws + r * pitch + ((16 * c) % NL) * lp + (16 * c) / NL;
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int q = 0; q < 16; ++q) to[q * lp] = (float)(int8_t)(w[q >> 2] >> (8 * (q & 3)));
        } else {
            float* const to = ws + r * pitch + ((4 * c) % NL) * lp + (4 * c) / NL;
            to[0] = __uint_as_float(v.x); to[lp] = __uint_as_float(v.y);
            to[2 * lp] = __uint_as_float(v.z); to[3 * lp] = __uint_as_float(v.w);
        }
    };
    auto put_row = [&](int i, const uint4& v) {
        const int r = xpr == 1 ? i : (int)__umulhi((uint32_t)i, xrecip), c = i - r * xpr;
        float f[XN];
        Vec16<XT>::widen(v, f);
        float* const to = xs + r * pitch + ((XN * c) % NL) * lp + (XN * c) / NL;
#pragma unroll
        for (int q = 0; q < XN; ++q) to[q * lp] = f[q];
        if (norm) {
            float4* const s4 = reinterpret_cast<float4*>(sq + r * sp + XN * c);
#pragma unroll
            for (int q = 0; q < XN / 4; ++q)
                s4[q] = make_float4(__fmul_rn(f[4 * q], f[4 * q]), __fmul_rn(f[4 * q + 1], f[4 * q + 1]),
                                    __fmul_rn(f[4 * q + 2], f[4 * q + 2]), __fmul_rn(f[4 * q + 3], f[4 * q + 3]));
        }
    };
    struct Six {
        uint4 v0, v1, v2, v3, v4, v5;
    };
    auto request = [&](const uint4* src, int n, int i) -> Six {  // pieces i, i + NT, ... (past the end: the last one)
        auto f = [&](int u) -> uint4 { return src[(uint32_t)min(i + u * NT, n - 1)]; };
        return Six{f(0), f(1), f(2), f(3), f(4), f(5)};
    };
    auto deliver = [&](const Six& s, int n, int i, auto put) {
        auto p = [&](int u, const uint4& v) {
            if (i + u * NT < n) put(i + u * NT, v);
        };
        p(0, s.v0); p(1, s.v1); p(2, s.v2); p(3, s.v3); p(4, s.v4); p(5, s.v5);
    };
    auto router_src = [&](int e0) {
        return NL == 32 ? reinterpret_cast<const uint4*>(a.wq + (size_t)e0 * d) : reinterpret_cast<const uint4*>(a.wr + (size_t)e0 * d);
    };
    auto rest_of_router = [&](int e0, int n, int from) {
        for (int i = from + tid; i < n; i += 6 * NT) deliver(request(router_src(e0), n, i), n, i, put_router);
    };
    // (the short last pieces' zeros)
    const int short_from = d / NL, short_n = (short_from + 3) / 4 * 4 - short_from;
    if (short_n > 0)
        for (int i = tid; i < TB * NL * short_n; i += NT) xs[(i / short_n) * lp + short_from + i % short_n] = 0.0f;
    const int nw0 = min(EG, e_to - e_from) * wpr, nx = nt * xpr;
    if (wave_norm) {
        // a wave a row: the raw elements in registers, normed, rounded to the layer's own type and laid down; each half of the
        // wave takes half of a lane's elements.  The router's rows are put into place meanwhile by whoever is free.
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = (tid >> 5) & 1;
        const XT* const rows = static_cast<const XT*>(a.x) + (size_t)t0 * d;
        with_lane_elements(d, [&](auto l_tag) {
            constexpr int L = decltype(l_tag)::value, H = L / 2;
            const int c0 = (tid & 31) * L + half * H;
            LaneRow<XT, L> row;
            row.load(rows + (size_t)min(wave, nt - 1) * d);
            float4 nwv[H / 4];
#pragma unroll
            for (int i = 0; i < H / 4; ++i) nwv[i] = *reinterpret_cast<const float4*>(a.norm_w + c0 + 4 * i);
            const Six w = request(router_src(e_from), nw0, tid);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
            for (int r = wave; r < nt; r += NT / 64) {
                const float inv_r = row.inverse_rms(a.norm_eps);
                float v[L];
                row.widen(v);
                if (r + NT / 64 < nt) row.load(rows + (size_t)(r + NT / 64) * d);
                float* const to = xs + r * pitch;
                XT o[H];
#pragma unroll
                for (int i = 0; i < H; ++i) {
                    const float4 n4 = nwv[i / 4];
                    const float n = i % 4 == 0 ? n4.x : i % 4 == 1 ? n4.y : i % 4 == 2 ? n4.z : n4.w;
                    o[i] = from_f32<XT>(__fmul_rn(__fmul_rn(half ? v[H + i] : v[i], inv_r), n));
                    const int c = c0 + i;
                    to[(c % NL) * lp + c / NL] = to_f32(o[i]);
                }
                auto put4 = [&](auto* base, int i) {  // four neighbours of the row in memory
                    typedef typename std::remove_pointer<decltype(base)>::type T;
                    T* const at = base + (size_t)(t0 + r) * d + c0 + 4 * i;
                    const float f[4] = {to_f32(o[4 * i]), to_f32(o[4 * i + 1]), to_f32(o[4 * i + 2]), to_f32(o[4 * i + 3])};
                    if constexpr (sizeof(T) == 4)
                        *reinterpret_cast<float4*>(at) = make_float4(f[0], f[1], f[2], f[3]);
                    else
                        *reinterpret_cast<uint2*>(at) = make_uint2(f32_to_bf16_bits(f[0]) | ((uint32_t)f32_to_bf16_bits(f[1]) << 16),
                                                                   f32_to_bf16_bits(f[2]) | ((uint32_t)f32_to_bf16_bits(f[3]) << 16));
                };
#pragma unroll
                for (int i = 0; i < H / 4; ++i) {
                    if (a.xn_out != nullptr) put4(static_cast<XT*>(a.xn_out), i);
                    if constexpr (sizeof(XT) == 4)
                        if (a.rows16 != nullptr) put4(a.rows16, i);
                }
            }
            deliver(w, nw0, tid, put_router);
            rest_of_router(e_from, nw0, 6 * NT);
        });
    } else {
        const uint4* const xsrc = reinterpret_cast<const uint4*>(static_cast<const XT*>(a.x) + (size_t)t0 * d);
        const Six w = request(router_src(e_from), nw0, tid);
        const Six x = request(xsrc, nx, tid);
        float nwv[2] = {0.0f, 0.0f};
        if (norm) {
            nwv[0] = a.norm_w[min(tid, d - 1)];
            nwv[1] = a.norm_w[min(tid + NT, d - 1)];
        }
        __builtin_amdgcn_sched_barrier(0);
        deliver(x, nx, tid, put_row);
        for (int i = tid + 6 * NT; i < nx; i += 6 * NT) deliver(request(xsrc, nx, i), nx, i, put_row);
        if (norm) {
            if (tid < d) nws[tid] = nwv[0];
            if (tid + NT < d) nws[tid + NT] = nwv[1];
            for (int c = tid + 2 * NT; c < d; c += NT) nws[c] = a.norm_w[c];
            __syncthreads();
            if (tid < nt) inv[tid] = inverse_rms_of(ordered_sum(sq + tid * sp, d), d, a.norm_eps);
            __syncthreads();
        }
        deliver(w, nw0, tid, put_router);
        rest_of_router(e_from, nw0, 6 * NT);
        if (short_n > 0)
            for (int i = tid; i < EG * NL * short_n; i += NT) ws[(i / short_n) * lp + short_from + i % short_n] = 0.0f;
    }
    if (!wave_norm && (norm || a.rows16 != nullptr)) {
        if (!norm) __syncthreads();
        // the normed rows, rounded to the layer's own type, replace the raw ones; they (and the bf16 copy of f32 rows
        // for the expert products) are written out on the way
        const int pieces = d / 8;
        const uint32_t recip = (uint32_t)(0x100000000ull / (uint32_t)pieces) + 1u;
        for (int i = tid; i < nt * pieces; i += NT) {
            const int r = pieces == 1 ? i : (int)__umulhi((uint32_t)i, recip), c = (i - r * pieces) * 8;
            float* const at = xs + r * pitch + (c % NL) * lp + c / NL;
            float v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = at[q * lp];
            if (norm) {
                const float sc = inv[r];
                const float4 wa = *reinterpret_cast<const float4*>(nws + c), wb = *reinterpret_cast<const float4*>(nws + c + 4);
                const float w[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
                XT o[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    o[q] = from_f32<XT>(__fmul_rn(__fmul_rn(v[q], sc), w[q]));
                    v[q] = to_f32(o[q]);
                    at[q * lp] = v[q];
                }
                if (a.xn_out != nullptr) {
                    uint4* const to = reinterpret_cast<uint4*>(static_cast<XT*>(a.xn_out) + (size_t)(t0 + r) * d + c);
#pragma unroll
                    for (int q = 0; q < 8 / XN; ++q) to[q] = reinterpret_cast<const uint4*>(o)[q];
                }
            }
            if constexpr (sizeof(XT) == 4) {
                if (a.rows16 != nullptr) {
                    uint4 o;
                    o.x = f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16);
                    o.y = f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16);
                    o.z = f32_to_bf16_bits(v[4]) | ((uint32_t)f32_to_bf16_bits(v[5]) << 16);
                    o.w = f32_to_bf16_bits(v[6]) | ((uint32_t)f32_to_bf16_bits(v[7]) << 16);
                    *reinterpret_cast<uint4*>(a.rows16 + (size_t)(t0 + r) * d + c) = o;
                }
            }
        }
    }
    __syncthreads();
    // ---- logits -------------------------------------------------------------------
    const int j = tid % NL;  // the thread's column lane
    const int quads = (d / NL + 3) / 4;
    for (int e0 = e_from; e0 < e_to; e0 += EG) {
        const int ne = min(EG, e_to - e0);
        if (e0 > e_from) {
            __syncthreads();  // the group before has been consumed
            rest_of_router(e0, ne * wpr, 0);
            __syncthreads();
        }
        const int etiles = (ne + EE - 1) / EE;
        const int tasks = (TB / TT) * etiles;
        for (int g0 = 0; g0 < tasks; g0 += NT / NL) {
            const int g = g0 + tid / NL;
            if (g0 + (int)(threadIdx.x & ~63u) / NL >= tasks) break;  // none of the wave's groups has a tile
            const int tt = min(g / etiles, TB / TT - 1), et = g - (g / etiles) * etiles;
            const unsigned char *xp[TT], *wp[EE];  // (a token or expert past the end: the last one's sums again, dropped)
#pragma unroll
            for (int u = 0; u < TT; ++u)
                xp[u] = reinterpret_cast<const unsigned char*>(xs + min(tt * TT + u, nt - 1) * pitch + j * lp);
#pragma unroll
            for (int u = 0; u < EE; ++u)
                wp[u] = reinterpret_cast<const unsigned char*>(ws + min(et * EE + u, ne - 1) * pitch + j * lp);
            float acc[TT][EE];
#pragma unroll
            for (int u = 0; u < TT; ++u)
#pragma unroll
                for (int v = 0; v < EE; ++v) acc[u][v] = 0.0f;
            struct Operands {
                float4 x[TT], w[EE];
            };
            // four steps of the chain a trip, the next trip's operands read before this one's products (two sets of
            // registers take turns)
            auto read = [&](Operands& o, int q) {
#pragma unroll
                for (int u = 0; u < TT; ++u) o.x[u] = lds_load_ahead<float4>(xp[u] + 16 * q);
#pragma unroll
                for (int u = 0; u < EE; ++u) o.w[u] = lds_load_ahead<float4>(wp[u] + 16 * q);
                __builtin_amdgcn_sched_barrier(0);
            };
            auto multiply = [&](const Operands& o) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int u = 0; u < TT; ++u)
#pragma unroll
                        for (int v = 0; v < EE; ++v)
                            acc[u][v] = __fadd_rn(acc[u][v], __fmul_rn(reinterpret_cast<const float*>(&o.x[u])[c],
                                                                       reinterpret_cast<const float*>(&o.w[v])[c]));
                __builtin_amdgcn_sched_barrier(0);
            };
            Operands oa, ob;
            read(oa, 0);
            int q = 0;
            for (; q + 2 <= quads; q += 2) {
                read(ob, q + 1);
                multiply(oa);
                read(oa, min(q + 2, quads - 1));
                multiply(ob);
            }
            if (q < quads) multiply(oa);
            // the column lanes folded left to right: lane l of a group holds ((0 + a_0) + a_1) + ... + a_l after l steps
            // of "take the lane below's sum, add your own" (see softmax_topk), the products side by side: one add a step,
            // where keeping a group's first lane apart took three instructions (32 column lanes, 8 tokens x 8 experts: 0.5 us)
            float own[TT][EE];
#pragma unroll
            for (int u = 0; u < TT; ++u)
#pragma unroll
                for (int v = 0; v < EE; ++v) {
                    own[u][v] = acc[u][v];
                    acc[u][v] = __fadd_rn(0.0f, acc[u][v]);
                }
            for (int st = 1; st < NL; ++st) {
#pragma unroll
                for (int u = 0; u < TT; ++u)
#pragma unroll
                    for (int v = 0; v < EE; ++v)
                        acc[u][v] = __fadd_rn(__uint_as_float(lanes_from<0x138>(__float_as_uint(acc[u][v]))), own[u][v]);  // wave_shr:1
            }
#pragma unroll
            for (int u = 0; u < TT; ++u)
#pragma unroll
                for (int v = 0; v < EE; ++v) {
                    const int t = tt * TT + u, el = et * EE + v, e = e0 + el;
                    if (j == NL - 1 && g < tasks && t < nt && el < ne) {
                        float y = __fadd_rn(acc[u][v], 0.0f);  // the reference adds its (empty) scalar rest: sum + 0
                        if constexpr (NL == 32) y = __fmul_rn(y, a.wscale[e]);
                        if (a.bias) y = __fadd_rn(y, a.bias[e]);
                        prob[t * ES + e] = y;
                    }
                }
        }
    }
}

}  // namespace rbmoe
