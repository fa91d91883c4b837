// Routing code shared by the large-batch and the decode-shaped kernels: norm, logits, softmax and top-k of a block of
// tokens whose rows lie in LDS as a whole.
#pragma once

#include "rbmoe_kernels.h"

namespace rbmoe {

// Dynamic LDS layout of router_kernel (floats / ints, in this order):
//   prob   [TB][ES]   logits, then probabilities   (ES = E | 1)
//   lsev   [TB]       log-sum-exp per token
//   lexp   [TB][k]    selected expert per local slot (-1 = unrouted)
//   wcount [waves][E] per-wave match counts of one ranking round
//   running[E]        slots already ranked per expert
__host__ __device__ static size_t router_fixed_bytes(int E, int k, int tokens = kRouterTokens) {
    const int ES = E | 1;
    size_t n = (size_t)tokens * ES + tokens + (size_t)tokens * k + (size_t)kRouterWaves * E + E;
    return (n * 4 + 15) & ~(size_t)15;
}

// The arrays that softmax and top-k leave for a block's tokens: in memory (of the whole call), and in LDS for what follows.
struct RouteOut {
    float* P;
    float* lse;
    int* expert_of;
    float* gate_of;
};

template <int I>
__device__ __forceinline__ float from_row_lane(float v) {  // lane I of each row of 16
    return __uint_as_float(lanes_from<0x150 + I>(__float_as_uint(v)));
}
// ((sum + v_FROM) + ...) + v_(TO - 1), v_i of lane i of the row, in every lane of the row
template <int FROM, int TO>
__device__ __forceinline__ float add_row_lanes(float sum, float v) {
    if constexpr (FROM == TO) return sum;
    else return add_row_lanes<FROM + 1, TO>(__fadd_rn(sum, from_row_lane<FROM>(v)), v);
}

// softmax, log-sum-exp and the k argmax rounds for the tokens of one wave of a router block (see router_tail), G lanes a
// token (16, 32 or 64: the least that E fits; lane j owns the experts j, j + G, ...).  `logit(token, expert)` gives the logits; probabilities, lse,
// experts and gates go to memory from the lanes that have them, and to `prob`, `lsev` and `lexp` for the ranks and losses.
// Everything order-sensitive keeps the reference's order: the maximum ignores NaN (f32::max), exp(v - max) is
// summed one expert after the other in index order, the k argmax rounds prefer the lower index on equal
// probabilities, and the gates are summed in rank order.
// The sum: a row of 16 lanes adds its lanes' exponentials one after the other, each handed to the whole row by the
// lane-permuting operand of the addition itself (row_newbcast); the next row goes on from there (lanes past the last expert
// add zeros).  An argmax round is a reduction of 32 bits - the greatest probability bits (probabilities are never negative, so the
// bits order like the values) - and a ballot for the lowest lane that holds them; a lane remembers the round that took it.
// NQ = turns a wave needs for its tokens (64 / G tokens a turn); the NQ turns share no data and run interleaved.
// A dependent chain from end to end.  G is a compile-time constant: with one of run time every step of a reduction was a branch,
// and with the sums shifted from lane to lane, gates divided in LDS and the results copied out behind a barrier the phase took
// 1.9 us for 8 experts and 2.2 for 16; now 1.0 and 1.1.  us a call, before / after: one row of the default model 12.8 / 12.2,
// 203 rows by 16 experts 47.6 / 46.9, 2048 rows of the default model 35.8 / 34.7, 8192 rows skewed 153.3 / 150.3.
template <int MAXJ, int NQ, int TB, int G, typename LOGIT>
__device__ __forceinline__ void softmax_topk(float* __restrict__ prob, float* __restrict__ lsev, int* __restrict__ lexp, int t0,
                                             int nt, int ES, const uint8_t* __restrict__ valid, int E, int k, const RouteOut& out,
                                             LOGIT&& logit) {
    constexpr int TW = TB < kRouterWaves ? 1 : TB / kRouterWaves;  // tokens of a wave
    const int lane_ = threadIdx.x & 63, wave_ = threadIdx.x >> 6;
    const int lig = lane_ & (G - 1);          // lane in group
    const int gbase = lane_ & ~(G - 1);       // first lane of the group
    constexpr int tpw = 64 / G;               // tokens a wave handles in one turn
    const unsigned long long gmask = (G == 64 ? ~0ull : ((1ull << (G & 63)) - 1ull)) << gbase;
    const unsigned long long below = gmask & ((1ull << lane_) - 1ull);  // the group's lower lanes
    const float neg_inf = __uint_as_float(0xff800000u);
    int tok[NQ];
    bool live[NQ], ok[NQ];
    float pv[NQ][MAXJ], mx[NQ], sum[NQ], total[NQ], lse[NQ];
    int taken[NQ][MAXJ];  // the round that took expert lig + G j, or -1
    uint8_t in_use[NQ];   // (asked for here, looked at behind the softmax)
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        tok[q] = wave_ * TW + q * tpw + lane_ / G;  // token of this group in turn q
        live[q] = tok[q] < nt && tok[q] < (wave_ + 1) * TW && q * tpw < TW;
        in_use[q] = valid != nullptr ? valid[t0 + (live[q] ? tok[q] : 0)] : 1;
        mx[q] = neg_inf;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int e = lig + G * j;
            pv[q][j] = (live[q] && e < E) ? logit(tok[q], e) : neg_inf;
            const float vv = (pv[q][j] == pv[q][j]) ? pv[q][j] : neg_inf;  // a NaN never becomes the maximum
            mx[q] = vv > mx[q] ? vv : mx[q];
            taken[q][j] = -1;
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) mx[q] = group_fmax(mx[q], G);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        sum[q] = 0.0f;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int e = lig + G * j;
            // lanes without an expert carry +0 through the sums below
            const float ex = rb_expf(__fadd_rn(pv[q][j], -mx[q]));
            pv[q][j] = (live[q] && e < E) ? ex : 0.0f;
        }
    }
    // the sums: one chain of adds per token in index order, row after row, slice after slice
#pragma unroll
    for (int j = 0; j < MAXJ; ++j) {
        if (MAXJ > 1 && G * j >= E) break;  // uniform
        auto row = [&](int r) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) sum[q] = add_row_lanes<0, 8>(sum[q], pv[q][j]);
            if (G * j + 16 * r + 8 < E)
#pragma unroll
                for (int q = 0; q < NQ; ++q) sum[q] = add_row_lanes<8, 16>(sum[q], pv[q][j]);
            if constexpr (G > 16)
#pragma unroll
                for (int q = 0; q < NQ; ++q) {  // row r's, to the whole group
                    const uint32_t lo = __builtin_amdgcn_readlane(__float_as_uint(sum[q]), 16 * r);
                    const uint32_t hi = G == 64 ? lo : __builtin_amdgcn_readlane(__float_as_uint(sum[q]), 32 + 16 * r);
                    sum[q] = __uint_as_float(G == 32 && (lane_ & 32) ? hi : lo);
                    asm("" : "+v"(sum[q]));  // (known to be the same in every lane it would be taken through scalar registers)
                }
        };
        const int rows = min(G / 16, (E - G * j + 15) / 16);
#pragma unroll 1
        for (int r = 0; r < rows; ++r) row(r);
    }
    bool any_nan = false;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        lse[q] = __fadd_rn(mx[q], rb_logf(sum[q]));
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const float share = __fdiv_rn(pv[q][j], sum[q]);
            pv[q][j] = sum[q] > 0.0f ? share : pv[q][j];
            any_nan = any_nan || pv[q][j] != pv[q][j];
        }
        ok[q] = live[q] && in_use[q] != 0;
        total[q] = 0.0f;
    }
    // ---- k rounds of argmax over the experts not yet taken ----
    // Without a NaN anywhere in the wave (with one expert a lane): the greatest probability bits among the untaken, then the
    // lowest of the lanes that hold them.
    if (MAXJ == 1 && __ballot(any_nan) == 0ull) {  // uniform over the wave
        for (int r = 0; r < k; ++r) {
            uint32_t best[NQ];
            bool open[NQ];  // this lane has an expert and it is not taken
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                open[q] = live[q] && lig < E && taken[q][0] < 0;
                best[q] = group_umax(open[q] ? __float_as_uint(pv[q][0]) : 0u, G);
            }
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const bool holds = open[q] && __float_as_uint(pv[q][0]) == best[q];
                const unsigned long long holders = __ballot(holds);
                taken[q][0] = holds && (holders & below) == 0ull ? r : taken[q][0];
                total[q] = __fadd_rn(total[q], __uint_as_float(best[q]));
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
                const unsigned long long m = __ballot(e < E && taken[q][j] < 0) & gmask;
                if (m != 0ull) first[q] = (__ffsll((long long)m) - 1 - gbase) + G * j;
            }
            // best candidate of this lane: not taken, not NaN; greater probability, then lower index
            has[q] = false;
            lbits[q] = 0;
            le[q] = 0x7fffffffu;
#pragma unroll
            for (int j = 0; j < MAXJ; ++j) {
                const int e = lig + G * j;
                if (live[q] && e < E && taken[q][j] < 0 && pv[q][j] == pv[q][j]) {
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
                    taken[q][j] = r;
                }
            // the winner's probability is the greatest bits themselves; only a NaN first expert has to be fetched
            float bestv = __uint_as_float(mbits[q]);
            if (__ballot(use_first) != 0ull) {  // uniform over the wave
                const float fv = __shfl(mine, gbase + (best & (G - 1)));
                if (use_first) bestv = fv;
            }
            total[q] = __fadd_rn(total[q], bestv);
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        if (live[q] && lig == 0) {
            lsev[tok[q]] = lse[q];
            out.lse[t0 + tok[q]] = lse[q];
        }
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int e = lig + G * j;
            if (!live[q] || e >= E) continue;
            prob[tok[q] * ES + e] = pv[q][j];
            out.P[(size_t)(t0 + tok[q]) * E + e] = pv[q][j];
            if (taken[q][j] < 0) continue;
            const int slot = tok[q] * k + taken[q][j];
            const float gate = total[q] > 0.0f ? __fdiv_rn(pv[q][j], total[q]) : pv[q][j];
            const int to = ok[q] ? e : -1;
            lexp[slot] = to;
            out.expert_of[(size_t)t0 * k + slot] = to;
            out.gate_of[(size_t)t0 * k + slot] = ok[q] ? gate : 0.0f;
        }
    }
}

// ... for the tokens of a whole block of TB, MAXJ = experts a lane may own: 1 when E <= 64
template <int MAXJ, int TB, typename LOGIT>
__device__ __forceinline__ void block_softmax_topk(float* prob, float* lsev, int* lexp, int t0, int nt, const uint8_t* valid, int E,
                                                   int k, const RouteOut& out, LOGIT&& logit) {
    // a wave's tokens (four of 32): all at once with 16 lanes per token, in more turns with 32 or 64 - the
    // turns are worked on side by side (one instruction stream), because each is a chain of dependent steps
    constexpr int TW = TB < kRouterWaves ? 1 : TB / kRouterWaves;
    const int ES = E | 1;
    if (MAXJ == 1 && E <= 16) softmax_topk<1, (TW + 3) / 4, TB, 16>(prob, lsev, lexp, t0, nt, ES, valid, E, k, out, logit);
    else if (MAXJ == 1 && E <= 32) softmax_topk<1, (TW + 1) / 2, TB, 32>(prob, lsev, lexp, t0, nt, ES, valid, E, k, out, logit);
    else softmax_topk<MAXJ, TW, TB, 64>(prob, lsev, lexp, t0, nt, ES, valid, E, k, out, logit);
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
    bool exact = false;     // route_exact_body takes the rows
    int slice = 0;          // route_rows_kernel: experts of a workgroup (0: all of them)
    int* arrive = nullptr;  // ... and, with a slice, a token block's arrival counter, kDecodeCombineCounterStride apart
    const int* exact_now = nullptr;  // RouterArgs::exact_now
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
            // of "take the lane below's sum, add your own" (a shift of the whole wave by one lane inside the add), the products side
            // by side.  A group's first lane takes in what the group below hands up, and wrong sums follow from there - one lane
            // behind the right ones, which nothing overtakes: after NL - 1 steps the last lane's is right.  One add a step, where
            // keeping a group's first lane apart took three instructions (32 column lanes, 8 tokens x 8 experts: 0.5 us)
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

// ---------------------------------------------------------------------------
// route_exact_body: what route_rows_body does, for bf16 rows and router weights whose products with them are exact
// (RouterArgs::exact, RowRange): there one fused multiply-add rounds as the reference's multiply and add do, and the f32
// matrix product of 16 x 16 x 4 is just that - its four columns one after the other, in index order, a fused multiply-add
// each (held against fmaf in every bit for bf16 and f32 operands, 5e4 sums) - so a column lane's sums run on the matrix cores, at
// four times the rate of a multiply and an add on the vector units and a sixteenth of their reads from LDS.
// Rows and router rows lie in LDS in bf16, column lane by column lane, and within one the 16 steps of a block so that lane
// (row, q) of the product finds its steps q, q + 4, q + 8, q + 12 in one 8-byte piece; who moves four pieces of a row there turns
// them over in registers.  Wave w owns the column lanes w NL / 8 ..; the lanes' sums meet in LDS and are folded left to right by
// a thread a logit.
// A token whose row holds an element out of RowRange gets its sums one multiply and one add at a time (rounded_sums), beside the
// products of its block.  So does every token of a launch that finds RouterArgs::exact_now unset, which a launch recorded under other
// weights does - over the weights in memory, for what is staged of them are bf16 parts.
// us a call with no such element / one in one row / one in every row: 203 tokens, d 768, 16 experts, behind a norm 27.2 / 29.3 / 32.3; 8192
// of them without 45.8 / 49.1 / 59.5; 16384, d 1024, 64 experts 213 / 225 / 346 (route_rows_body or logits_kernel: 28.8, 50.4, 270, whatever
// the elements).  The routing alone under weights that were set after the launch was recorded, beside a launch chosen for them: 10.7
// against 8.0, 22.3 against 14.2, 165 against 89.
// Bound by the length of a workgroup's chain, not by work: 203 tokens, d 768, 16 experts, behind a norm, from the kernel's start:
// normed rows laid down at 2.6 us, every wave's rows and weights at 3.7, sums 5.2, met 5.6, softmax and top-k 6.8, end 7.6; 8192
// tokens without a norm 3.2, 3.7, 6.0, 6.7, 7.9, 8.7 (route_rows_body, with the same tail: 10.1 less the tail's 1.2; 11.7).  us a
// call, route_rows_body / this: the two 48.4 / 47.6 and 157.3 / 153.3, 4096 tokens by 8 experts (int8) 91.3 / 89.8, 2048 of d 512
// behind a norm 36.5 / 35.8.
// ---------------------------------------------------------------------------
// Elements of bf16 rows: nothing but zeros and magnitudes from 2^-72 to below 2^80.  Two at a time, as the bits lie in memory.
struct RowRange {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    u16x2 most = {0, 0}, least = {0xffff, 0xffff};  // of the magnitudes' bits; of the same less one, zeros aside
    __device__ __forceinline__ void see(uint32_t two) {
        const u16x2 m = __builtin_bit_cast(u16x2, two & 0x7fff7fffu);
        most = __builtin_elementwise_max(most, m);
        least = __builtin_elementwise_min(least, m - (u16x2){1, 1});
    }
    __device__ __forceinline__ void see(const uint4& v) { see(v.x); see(v.y); see(v.z); see(v.w); }
    __device__ __forceinline__ bool left() const {
        return max(most.x, most.y) >= ((127 + 80) << 7) || min(least.x, least.y) < ((127 - 72) << 7) - 1;
    }
};

typedef float floatx4 __attribute__((ext_vector_type(4)));

__host__ __device__ static int exact_lane_steps(int d, int NL) { return (d / NL + 15) & ~15; }
// Bytes of a staged row: 16 rows' pieces of the same step start in different banks.
__host__ __device__ static int exact_row_bytes(int d, int NL) { return NL * exact_lane_steps(d, NL) * 2 + 16; }
// Experts whose column lanes' sums meet in LDS at a time.
__host__ __device__ constexpr int exact_round(int TB, int NL) { return TB * NL > 512 ? 8 : 16; }
// Whether route_exact_body takes the call's rows (which lie on 16-byte boundaries, in whole turns of the column lanes).
__host__ static inline bool route_exact_ok(const RouterArgs& a, bool bf16) {
    return bf16 && a.exact && a.rows16 == nullptr && (!a.norm_w || wave_norms(a.d));
}
// The next smaller number of experts whose rows may lie in LDS together: whole rounds.
__host__ static inline int exact_fewer(int EG, int TB, int NL) { return (EG - 1) / exact_round(TB, NL) * exact_round(TB, NL); }
__host__ __device__ static size_t route_exact_lds_bytes(int E, int k, int d, int TB, int NL, int EG) {
    return router_fixed_bytes(E, k, TB) + 4 * kRouterWaves + (size_t)NL * TB * exact_round(TB, NL) * 4 +
           (size_t)(TB + EG) * exact_row_bytes(d, NL);
}

// The column lanes' sums of one token and expert, folded left to right; `part`: lane 0's.
template <int TB, int NL>
__device__ __forceinline__ float fold_lanes(const float* part) {
    float v[NL], y = 0.0f;
#pragma unroll
    for (int l = 0; l < NL; ++l) v[l] = part[l * TB * exact_round(TB, NL)];
#pragma unroll
    for (int l = 0; l < NL; ++l) y = __fadd_rn(y, v[l]);
    return __fadd_rn(y, 0.0f);  // the reference adds its (empty) scalar rest: sum + 0
}

// The column lanes' sums of `ne` experts from e0 on into `part`, for the tokens whose bits are set, one multiply and one add at a
// time: token rows as they are staged, the router's weights from memory - a thread's sixteen of a block of steps serve up to four
// tokens, the same for a whole wave, which leaves out those without a bit.  Bound by the vector units and the wait for the weights.
// What counts first is that the kernels around it stay small: with eight tokens a thread (37.5 KB and 118 registers instead of 35.8 and
// 106) 16384 tokens of d 1024 by 64 experts are rounded 6 % faster, but 9000 of d 512 by 8, none of them rounded, are routed in 13.1 us
// instead of 12.5; with the weights asked for a block ahead the kernels take 150 to 190 registers.
template <int TB, int NL>
__device__ __forceinline__ void rounded_sums(const RouteRowsArgs& a, const unsigned char* xs, float* part, uint32_t tokens, int nt, int e0,
                                             int ne) {
    constexpr int RE = exact_round(TB, NL), TT = TB * RE * NL / kRouterThreads < 4 ? 2 : 4;
    const int S = a.d / NL, Sp = exact_lane_steps(a.d, NL), pitch = exact_row_bytes(a.d, NL);
#pragma unroll 1
    for (int i = threadIdx.x; i < (TB / TT) * RE * NL; i += kRouterThreads) {
        const int j = i % NL, e = i / NL % RE, t = i / (NL * RE) * TT;
        if (e >= ne || ((tokens >> t) & ((1u << TT) - 1)) == 0) continue;
        const unsigned char* x[TT];
#pragma unroll
        for (int u = 0; u < TT; ++u) x[u] = xs + min(t + u, nt - 1) * pitch + j * Sp * 2;
        float sum[TT] = {};
        struct Steps {
            float w[16];
        };
        const size_t row = (size_t)(e0 + e) * a.d + j;
        auto weight = [&](size_t at) -> float {
            if constexpr (NL == 32) return (float)a.wq[at];
            else return a.wr[at];
        };
        auto add = [&](const Steps& v, int s0) {
#pragma unroll
            for (int u = 0; u < TT; ++u) {
                if (((tokens >> (t + u)) & 1u) == 0) continue;
                const uint4 lo = *reinterpret_cast<const uint4*>(x[u] + 2 * s0), hi = *reinterpret_cast<const uint4*>(x[u] + 2 * s0 + 16);
                const uint32_t two[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                for (int s = 0; s < 16; ++s) {
                    const int p = (s & 3) * 4 + (s >> 2);
                    const float f = __uint_as_float(p & 1 ? two[p >> 1] & 0xffff0000u : two[p >> 1] << 16);
                    sum[u] = __fadd_rn(sum[u], __fmul_rn(f, v.w[s]));
                }
            }
        };
#pragma unroll 1
        for (int s0 = 0; s0 < S; s0 += 16) {
            Steps v;
            const size_t from = row + NL * s0;
            if (s0 + 16 <= S) {
#pragma unroll
                for (int s = 0; s < 16; ++s) v.w[s] = weight(from + NL * s);
            } else {  // (rows hold zeros past their end)
#pragma unroll
                for (int s = 0; s < 16; ++s) v.w[s] = s0 + s < S ? weight(from + NL * s) : 0.0f;
            }
            add(v, s0);
        }
#pragma unroll
        for (int u = 0; u < TT; ++u)
            if ((tokens >> (t + u)) & 1u) part[(j * TB + t + u) * RE + e] = sum[u];
    }
}

// With `fold_later` and one round of experts the sums are left where they meet (behind a barrier), for ExactLogits, and the result is
// true; otherwise the logits lie in `prob` and the caller meets at a barrier before it reads them.
template <int TB, int NL, bool NORM>
__device__ __forceinline__ bool route_exact_body(const RouteRowsArgs& a, int blk, int e_from, int e_to, bool fold_later,
                                                 unsigned char* __restrict__ lds_raw) {
    constexpr int NT = kRouterThreads, LW = NL / 8, MB = (TB + 15) / 16, RE = exact_round(TB, NL);
    const int T = a.T, d = a.d, E = a.E, k = a.k, EG = a.EG, ES = E | 1;
    float* const prob = reinterpret_cast<float*>(lds_raw);
    int* const left = reinterpret_cast<int*>(lds_raw + router_fixed_bytes(E, k, TB));  // [waves] elements out of RowRange
    float* const part = reinterpret_cast<float*>(left + kRouterWaves);                 // [NL][TB][RE]
    const int S = d / NL, Sp = exact_lane_steps(d, NL), pitch = exact_row_bytes(d, NL);
    unsigned char* const xs = reinterpret_cast<unsigned char*>(part + NL * TB * RE);
    unsigned char* const ws = xs + TB * pitch;
    const int tid = threadIdx.x, t0 = blk * TB, nt = min(TB, T - t0);
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int exact_now = 1;
    // (a vector load among the rows': a scalar one would be waited for with the kernel's arguments)
    auto ask_router = [&] {
        int zero = 0;
        asm("" : "+v"(zero));
        if constexpr (NL == 8)
            if (a.exact_now != nullptr) exact_now = a.exact_now[zero];
    };

    // Staging.  A piece is eight neighbouring columns; a task four pieces of a row, the steps 16 Q + 4 i + q.  (Past the end of
    // a row: zeros, which sums do not see.)
    constexpr int JB = NL / 8;  // pieces of a step
    const int per_row = Sp / 4 * JB;
    const uint32_t recip = (uint32_t)(0x100000000ull / (uint32_t)per_row) + 1u;  // exact for the few thousand tasks there are
    struct Task {
        int row, step, jb;  // its first step
        unsigned at;        // bytes from the row's start in LDS
    };
    auto task = [&](int i) {
        Task t;
        t.row = (int)__umulhi((uint32_t)i, recip);
        const int r = i - t.row * per_row, q = r / JB;  // 4 Q + q
        t.jb = r % JB;
        t.step = 16 * (q >> 2) + (q & 3);
        t.at = (unsigned)(8 * t.jb * Sp * 2 + 8 * q);
        return t;
    };
    auto turn = [&](unsigned char* to, const uint4 (&p)[4]) {  // p[i]: eight columns of step i, as bf16
        const uint32_t w[4][4] = {{p[0].x, p[0].y, p[0].z, p[0].w}, {p[1].x, p[1].y, p[1].z, p[1].w},
                                  {p[2].x, p[2].y, p[2].z, p[2].w}, {p[3].x, p[3].y, p[3].z, p[3].w}};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t pick = j & 1 ? 0x07060302u : 0x05040100u;
            const uint2 v = make_uint2(__builtin_amdgcn_perm(w[1][j >> 1], w[0][j >> 1], pick),
                                       __builtin_amdgcn_perm(w[3][j >> 1], w[2][j >> 1], pick));
            *reinterpret_cast<uint2*>(to + j * Sp * 2) = v;
        }
    };
    const uint4 zero = make_uint4(0, 0, 0, 0);
    struct Weights {  // a task's columns as they lie in memory
        uint4 v[NL == 32 ? 2 : 8];
    };
    auto weights_of = [&](int e0, int n, int i) {  // (past the end: the last task again)
        const Task t = task(min(i, n - 1));
        Weights w;
        if constexpr (NL == 32) {
            uint2 h[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                h[u] = *reinterpret_cast<const uint2*>(a.wq + (size_t)(e0 + t.row) * d + 32 * min(t.step + 4 * u, S - 1) + 8 * t.jb);
            w.v[0] = make_uint4(h[0].x, h[0].y, h[1].x, h[1].y);
            w.v[1] = make_uint4(h[2].x, h[2].y, h[3].x, h[3].y);
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint4* const from = reinterpret_cast<const uint4*>(a.wr + (size_t)(e0 + t.row) * d + 8 * min(t.step + 4 * u, S - 1));
                w.v[2 * u] = from[0];
                w.v[2 * u + 1] = from[1];
            }
        }
        return w;
    };
    auto put_weights = [&](int n, int i, unsigned char* to, const Weights& w) {
        if (i >= n) return;
        const Task t = task(i);
        uint4 p[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if constexpr (NL == 32) {
                const uint4& v = w.v[u >> 1];
                const uint2 h = u & 1 ? make_uint2(v.z, v.w) : make_uint2(v.x, v.y);
                p[u] = make_uint4(widen2(h.x, 0), widen2(h.x, 16), widen2(h.y, 0), widen2(h.y, 16));
            } else {
                const uint4 &lo = w.v[2 * u], &hi = w.v[2 * u + 1];  // (bf16 values: the lower halves are zero)
                p[u] = make_uint4(__builtin_amdgcn_perm(lo.y, lo.x, 0x07060302u), __builtin_amdgcn_perm(lo.w, lo.z, 0x07060302u),
                                  __builtin_amdgcn_perm(hi.y, hi.x, 0x07060302u), __builtin_amdgcn_perm(hi.w, hi.z, 0x07060302u));
            }
            if (t.step + 4 * u >= S) p[u] = zero;
        }
        turn(to + t.row * pitch + t.at, p);
    };
    auto rest_of_router = [&](int e0, int n, int from, unsigned char* to) {
        for (int i = from + tid; i < n; i += NT) put_weights(n, i, to, weights_of(e0, n, i));
    };
    const int nw0 = min(EG, e_to - e_from) * per_row;
    RowRange range;
    if constexpr (NORM) {
        // as in route_rows_body: a wave a row, each half of the wave half of a lane's elements (the widths of wave_norms)
        const int half = (tid >> 5) & 1;
        const bf16_t* const rows = static_cast<const bf16_t*>(a.x) + (size_t)t0 * d;
        with_lane_elements(d, [&](auto l_tag) {
            constexpr int L = decltype(l_tag)::value, H = L / 2;
            const int c0 = (tid & 31) * L + half * H;
            LaneRow<bf16_t, L> row;
            row.load(rows + (size_t)min(wave, nt - 1) * d);
            float4 nwv[H / 4];
#pragma unroll
            for (int i = 0; i < H / 4; ++i) nwv[i] = *reinterpret_cast<const float4*>(a.norm_w + c0 + 4 * i);
            const Weights w = weights_of(e_from, nw0, tid);
            ask_router();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
            for (int r = wave; r < nt; r += NT / 64) {
                const float inv_r = row.inverse_rms(a.norm_eps);
                float v[L];
                row.widen(v);
                if (r + NT / 64 < nt) row.load(rows + (size_t)(r + NT / 64) * d);
                uint32_t o[H / 2];
#pragma unroll
                for (int i = 0; i < H; i += 2) {
                    uint32_t two = 0;
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const float4 n4 = nwv[(i + u) / 4];
                        const float n = (i + u) % 4 == 0 ? n4.x : (i + u) % 4 == 1 ? n4.y : (i + u) % 4 == 2 ? n4.z : n4.w;
                        const uint32_t b = f32_to_bf16_bits(__fmul_rn(__fmul_rn(half ? v[H + i + u] : v[i + u], inv_r), n));
                        two |= b << (16 * u);
                        const int c = c0 + i + u, t = c / NL, j = c % NL;
                        *reinterpret_cast<uint16_t*>(xs + r * pitch + (j * Sp + (t & ~15) + (t & 3) * 4 + ((t >> 2) & 3)) * 2) = (uint16_t)b;
                    }
                    range.see(two);
                    o[i / 2] = two;
                }
                if (a.xn_out != nullptr) {
                    bf16_t* const to = static_cast<bf16_t*>(a.xn_out) + (size_t)(t0 + r) * d + c0;
#pragma unroll
                    for (int i = 0; i < H / 4; ++i) *reinterpret_cast<uint2*>(to + 4 * i) = make_uint2(o[2 * i], o[2 * i + 1]);
                }
            }
            put_weights(nw0, tid, ws, w);
        });
        // (a row's steps past its end)
        if (S < Sp)
            for (int i = tid; i < TB * NL * (Sp - S); i += NT) {
                const int q = i / (Sp - S), t = S + i % (Sp - S);
                *reinterpret_cast<uint16_t*>(xs + (q / NL) * pitch + ((q % NL) * Sp + (t & ~15) + (t & 3) * 4 + ((t >> 2) & 3)) * 2) = 0;
            }
    } else {
        const bf16_t* const rows = static_cast<const bf16_t*>(a.x) + (size_t)t0 * d;
        const int nx = nt * per_row;
        struct Rows {
            uint4 v[4];
        };
        auto rows_of = [&](int i) {
            const Task t = task(min(i, nx - 1));
            Rows r;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                r.v[u] = *reinterpret_cast<const uint4*>(rows + (size_t)t.row * d + NL * min(t.step + 4 * u, S - 1) + 8 * t.jb);
            return r;
        };
        auto put_rows = [&](int i, Rows r) {
            if (i >= nx) return;
            const Task t = task(i);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (t.step + 4 * u >= S) r.v[u] = zero;
                range.see(r.v[u]);
            }
            turn(xs + t.row * pitch + t.at, r.v);
        };
        // (two tasks a thread requested before the first is turned over, then the router's)
        Rows r0 = rows_of(tid), r1 = r0;
        if (NT < nx) r1 = rows_of(tid + NT);
        const Weights w = weights_of(e_from, nw0, tid);
        ask_router();
        __builtin_amdgcn_sched_barrier(0);
        put_rows(tid, r0);
        put_rows(tid + NT, r1);
        for (int i = tid + 2 * NT; i < nx; i += NT) put_rows(i, rows_of(i));
        put_weights(nw0, tid, ws, w);
    }
    rest_of_router(e_from, nw0, NT, ws);
    {
        const bool any = __ballot(range.left() || exact_now == 0) != 0ull;
        if (lane == 0) left[wave] = any;
    }
    __syncthreads();
    const bool router_exact = __builtin_amdgcn_readfirstlane(exact_now) != 0;
    int votes = 0;  // (all of them asked for before the first is looked at)
#pragma unroll
    for (int w = 0; w < kRouterWaves; ++w) votes |= left[w];
    uint32_t rounded = 0;  // the tokens whose sums are taken one rounding at a time
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(votes) != 0, 0)) {  // uniform over the workgroup
        __syncthreads();   // everyone has read the votes
        uint32_t mine = router_exact ? 0u : 0xffffffffu;
        if (router_exact)
            for (int t = wave; t < nt; t += kRouterWaves) {
                RowRange of_row;
                for (int i = lane; i < NL * Sp / 8; i += 64) of_row.see(*reinterpret_cast<const uint4*>(xs + t * pitch + 16 * i));
                mine |= __ballot(of_row.left()) != 0ull ? 1u << t : 0u;
            }
        if (lane == 0) left[wave] = (int)mine;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kRouterWaves; ++w) rounded |= (uint32_t)left[w];
        rounded = __builtin_amdgcn_readfirstlane(rounded);
    }
    // ---- the column lanes' sums, 16 (RE) experts at a time ----------------------------
    // Experts past the EG whose rows lie in LDS follow round by round, into the place of the round that is done with, asked for in
    // front of its products.
    const int blocks = (S + 15) / 16, last = (S - 16 * (blocks - 1) + 3) / 4;  // products of the last block of steps
    const int n = e_to - e_from;
    int room = 0;  // where the round's router rows lie
    for (int r0 = 0; r0 < n; r0 += RE) {
        const int ne = min(RE, n - r0), next = min(RE, n - r0 - EG);  // (next: experts that follow into its place)
        if (r0 > 0) __syncthreads();  // the round before has been folded, this one's rows are there
        Weights follow;
        if (next > 0) follow = weights_of(e_from + r0 + EG, next * per_row, tid);
        float scale = 1.0f, bias = 0.0f;  // of the expert whose logits this thread folds
        {
            const int e = min(e_from + r0 + tid % RE, e_to - 1);
            if constexpr (NL == 32) scale = a.wscale[e];
            if (a.bias) bias = a.bias[e];
        }
        __builtin_amdgcn_sched_barrier(0);
        unsigned char* const wr = ws + room * pitch;
        {
            if (router_exact) {  // uniform over the launch
                const unsigned char* x[MB];
                const unsigned at = (unsigned)(wave * LW * Sp * 2 + 8 * (lane >> 4));
#pragma unroll
                for (int b = 0; b < MB; ++b) x[b] = xs + min(16 * b + (lane & 15), nt - 1) * pitch + at;
                const unsigned char* const w = wr + min(lane & 15, ne - 1) * pitch + at;
                floatx4 acc[LW][MB];
#pragma unroll
                for (int u = 0; u < LW; ++u)
#pragma unroll
                    for (int b = 0; b < MB; ++b) acc[u][b] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                struct Operands {
                    uint2 x[LW][MB], w[LW];
                };
                auto read = [&](int Q) {
                    Operands o;
#pragma unroll
                    for (int u = 0; u < LW; ++u) {
                        o.w[u] = *reinterpret_cast<const uint2*>(w + u * Sp * 2 + 32 * Q);
#pragma unroll
                        for (int b = 0; b < MB; ++b) o.x[u][b] = *reinterpret_cast<const uint2*>(x[b] + u * Sp * 2 + 32 * Q);
                    }
                    return o;
                };
                auto multiply = [&](const Operands& o, int n) {
                    auto value = [](const uint2& v, int i) {
                        const uint32_t two = i < 2 ? v.x : v.y;
                        return __uint_as_float(i & 1 ? two & 0xffff0000u : two << 16);
                    };
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (i < n)
#pragma unroll
                            for (int u = 0; u < LW; ++u)
#pragma unroll
                                for (int b = 0; b < MB; ++b)
                                    acc[u][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(value(o.x[u][b], i), value(o.w[u], i), acc[u][b], 0, 0, 0);
                };
                Operands o = read(0);
                for (int Q = 0; Q + 1 < blocks; ++Q) {
                    const Operands next = read(Q + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    multiply(o, 4);
                    o = next;
                }
                multiply(o, last);
                // lane l holds the sums of the tokens 4 (l / 16) .. + 3 (of a block of 16) and expert l % 16
#pragma unroll
                for (int u = 0; u < LW; ++u)
#pragma unroll
                    for (int b = 0; b < MB; ++b)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int t = 16 * b + 4 * (lane >> 4) + i, e = lane & 15;
                            if (t < TB && e < ne) part[((wave * LW + u) * TB + t) * RE + e] = acc[u][b][i];
                        }
            }
            if (__builtin_expect(rounded != 0, 0)) {  // uniform over the workgroup
                if (router_exact) __syncthreads();  // these take the place of the products' sums
                rounded_sums<TB, NL>(a, xs, part, rounded, nt, e_from + r0, ne);
            }
            __syncthreads();
            if (fold_later && n <= RE) return true;
            if (next > 0) {
                put_weights(next * per_row, tid, wr, follow);
                rest_of_router(e_from + r0 + EG, next * per_row, NT, wr);
            }
            room = room + RE < EG ? room + RE : 0;
            static_assert(NT % RE == 0, "a thread folds one expert");
            for (int i = tid; i < nt * RE; i += NT) {
                const int t = i / RE, e = e_from + r0 + i % RE;
                if (i % RE >= ne) continue;
                float y = fold_lanes<TB, NL>(part + i);
                if constexpr (NL == 32) y = __fmul_rn(y, scale);
                if (a.bias) y = __fadd_rn(y, bias);
                prob[t * ES + e] = y;
            }
        }
    }
    return false;
}

// The logits behind route_exact_body, for a wave whose lane 16 g + e asks for expert e (or, folded already, any): what is added to or
// multiplied with the sums is asked for when the object is made.
template <int TB, int NL>
struct ExactLogits {
    const float *part, *prob;
    int ES;
    float scale = 1.0f, bias = 0.0f;
    bool has_bias, folded = false;
    __device__ __forceinline__ ExactLogits(const RouteRowsArgs& a, unsigned char* lds_raw) {
        prob = reinterpret_cast<const float*>(lds_raw);
        part = reinterpret_cast<const float*>(lds_raw + router_fixed_bytes(a.E, a.k, TB)) + kRouterWaves;
        ES = a.E | 1;
        const int e = min((int)threadIdx.x & 15, a.E - 1);
        has_bias = a.bias != nullptr;
        if (has_bias) bias = a.bias[e];
        if constexpr (NL == 32) scale = a.wscale[e];
    }
    __device__ __forceinline__ float operator()(int t, int e) const {
        if (folded) return prob[t * ES + e];  // uniform over the workgroup
        float y = fold_lanes<TB, NL>(part + t * exact_round(TB, NL) + e);
        if constexpr (NL == 32) y = __fmul_rn(y, scale);
        return has_bias ? __fadd_rn(y, bias) : y;
    }
};

// router_tail: everything behind the logits for the TB tokens of router block `blk` - softmax, log-sum-exp, top-k,
// gates, ranks, block histogram, partial sums of the losses.  `logit(token, expert)` may be read already.
// MAXJ = experts a lane may own: 1 when E <= 64 (a lane owns one expert), kMaxExperts / 64 otherwise.
template <int MAXJ, int TB, typename LOGIT>
__device__ __forceinline__ void router_tail(unsigned char* __restrict__ lds_raw, int blk, const uint8_t* __restrict__ valid, int T,
                                            int E, int k, const RouteOut& out, int* __restrict__ rank_in_block,
                                            int* __restrict__ blockcnt, float* __restrict__ partial, LOGIT&& logit) {
    const int ES = E | 1;
    float* prob = reinterpret_cast<float*>(lds_raw);
    float* lsev = prob + TB * ES;
    int* lexp = reinterpret_cast<int*>(lsev + TB);
    int* wcount = lexp + TB * k;
    int* running = wcount + kRouterWaves * E;

    const int tid = threadIdx.x;
    const int t0 = blk * TB;
    const int nt = min(TB, T - t0);
    const int nls = nt * k, rank_waves = (nls + 63) >> 6;
    for (int idx = tid; idx < E; idx += kRouterThreads) running[idx] = 0;
    if (rank_waves < kRouterWaves)
        for (int idx = tid; idx < rank_waves * E; idx += kRouterThreads) wcount[idx] = 0;
    block_softmax_topk<MAXJ, TB>(prob, lsev, lexp, t0, nt, valid, E, k, out, logit);
    __syncthreads();

    const int lane = tid & 63;
    const int wave = tid >> 6;
    int ebits = 0;
    while ((1 << ebits) < E) ++ebits;
    // the slot's lower lanes with its expert, and (in the first of them) how many lanes have it
    auto rank_in_wave = [&](int e, int& group) {
        unsigned long long mask = __ballot(e >= 0);
        for (int b = 0; b < ebits; ++b) {
            const bool bit = (e >> b) & 1;
            const unsigned long long bb = __ballot(bit);
            mask &= bit ? bb : ~bb;
        }
        group = __popcll(mask);
        return __popcll(mask & ((1ull << lane) - 1ull));
    };
    // ---- partial sums for the auxiliary losses (fixed order), by the threads from `first` on ----
    auto partial_sums = [&](int first) {
        for (int e = tid - first; e >= 0 && e <= E; e += kRouterThreads - first) {
            float s = 0.0f;
            for (int i0 = 0; i0 < nt; i0 += 8) {
                float pvv[8];
                int okv[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int i = min(i0 + u, nt - 1);
                    okv[u] = lexp[i * k];
                    pvv[u] = e < E ? prob[i * ES + e] : lsev[i] * lsev[i];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (i0 + u < nt && okv[u] >= 0) s += pvv[u];
            }
            partial[(size_t)blk * (E + 1) + e] = s;
        }
    };
    // ---- rank of every local slot among earlier slots of the same expert: the block's slots in a few waves, the others take
    // the partial sums meanwhile (64 experts, six a token: 5.3 us behind the softmax with one after the other) ----
    if (rank_waves < kRouterWaves) {
        const int ls = tid, e = ls < nls ? lexp[ls] : -1;
        int group = 0, rank = 0;
        if (wave < rank_waves) {  // uniform over the wave
            rank = rank_in_wave(e, group);
            if (e >= 0 && rank == 0) wcount[wave * E + e] = group;
        } else {
            partial_sums(64 * rank_waves);
        }
        if (rank_waves > 1) {
            __syncthreads();
        } else {
            if (wave != 0) return;
            __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's LDS writes have landed
            __builtin_amdgcn_wave_barrier();
        }
        if (e >= 0) {
            for (int w = 0; w < wave; ++w) rank += wcount[w * E + e];
            rank_in_block[(size_t)t0 * k + ls] = rank;
        }
        for (int idx = tid; idx < E; idx += rank_waves > 1 ? kRouterThreads : 64) {
            int count = 0;
            for (int w = 0; w < rank_waves; ++w) count += wcount[w * E + idx];
            blockcnt[(size_t)blk * E + idx] = count;
        }
        return;
    }
    partial_sums(0);
    const int rounds = (nls + kRouterThreads - 1) / kRouterThreads;
    for (int rd = 0; rd < rounds; ++rd) {
        for (int idx = tid; idx < kRouterWaves * E; idx += kRouterThreads) wcount[idx] = 0;
        __syncthreads();
        const int ls = rd * kRouterThreads + tid;
        const int e = (ls < nls) ? lexp[ls] : -1;
        int group;
        const int rank_w = rank_in_wave(e, group);
        if (e >= 0 && rank_w == 0) wcount[wave * E + e] = group;
        __syncthreads();
        if (e >= 0) {
            int pre = running[e];
            for (int w = 0; w < wave; ++w) pre += wcount[w * E + e];
            rank_in_block[(size_t)t0 * k + ls] = pre + rank_w;
        }
        __syncthreads();
        for (int idx = tid; idx < E; idx += kRouterThreads)
            for (int w = 0; w < kRouterWaves; ++w) running[idx] += wcount[w * E + idx];
        __syncthreads();
    }
    for (int idx = tid; idx < E; idx += kRouterThreads) blockcnt[(size_t)blk * E + idx] = running[idx];
}

// A token block's experts shared out over workgroups: each leaves its logits in P; the last to arrive fetches the others' into
// its own array and goes on.  Device-scope stores and loads: the workgroups may sit on different XCDs, whose L2s do not see
// each other's lines; a workgroup's stores are acknowledged before its arrival is counted.
template <int TB>
__device__ __forceinline__ bool last_slice(const RouteRowsArgs& a, int from, int to, unsigned char* lds_raw) {
    float* const prob = reinterpret_cast<float*>(lds_raw);
    const int E = a.E, ES = E | 1, tid = threadIdx.x;
    int& last = *reinterpret_cast<int*>(prob + TB * ES);  // (where router_tail will keep the log-sum-exps)
    const int t0 = blockIdx.x * TB, nt = min(TB, a.T - t0), n = to - from;
    for (int i = tid; i < nt * n; i += kRouterThreads) {
        const int t = i / n, e = from + i - t * n;
        __hip_atomic_store(a.P + (size_t)(t0 + t) * E + e, prob[t * ES + e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
        int* const counter = a.arrive + blockIdx.x * kDecodeCombineCounterStride;
        const int before = atomicAdd(counter, 1);
        last = before == (int)gridDim.y - 1;
        if (before == (int)gridDim.y - 1) atomicExch(counter, 0);  // everyone has arrived: ready for the next launch
    }
    __syncthreads();
    if (!last) return false;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    for (int i = tid; i < nt * E; i += kRouterThreads) {
        const int t = i / E, e = i - t * E;
        if (e < from || e >= to)
            prob[t * ES + e] = __hip_atomic_load(a.P + (size_t)t0 * E + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    return true;
}

hipError_t launch_route_exact(const RouterArgs& a, const RouterPlan& p, hipStream_t s);  // (route_exact.hip)

}  // namespace rbmoe
