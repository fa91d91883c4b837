// Decode-shaped forward (a few tokens): the layer is bound by streaming the touched experts'
// weights once from HBM and by launch latency.  The work is cut into four launches
//
//   route_small_kernel   one workgroup: logits, softmax, top-k, counting sort, tile table,
//                        auxiliary losses (MoeLayer::forward_train, src/moe.rs:243-341, up to
//                        the bucket loop; route src/moe.rs:553-593; losses src/moe.rs:325-337)
//   decode_gemm_kernel   gate/up + SwiGLU of every routed tile and of the shared expert
//   decode_gemm_kernel   down product of both
//   combine              (the same kernel as the large path)
//
// which the layer folds into fewer where the call allows it: the combine into the down launch (the last
// workgroup of a block of output columns to finish sums it), and - where fetching the untouched experts' weights too
// costs less than it saves - the routing into the gate/up launch (decode_front_kernel), behind which the down launch has one row of
// workgroups per expert (decode_down_by_expert_kernel) or, for a row or two, takes a column block's rows in one workgroup
// (decode_down_few_kernel): two launches.  The products are spread over (tile,
// 32-feature block) workgroups whose waves split the reduction dimension, so that a few hundred kilobytes of
// weight fragments are in flight per CU and every byte of a touched expert is fetched exactly once per 32-row tile.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "routing_device.h"

namespace rbmoe {

// ---------------------------------------------------------------------------
// route_small_kernel.  Everything is written the way the reference walks it, one token or
// one expert per thread, because at this size the order of operations matters and the time
// does not: logits in the order of the eight-lane `dot` (src/matrix.rs:26-40) with the
// eight lanes of a pair on eight neighbouring threads, softmax_rows and route per token,
// the bucket loop per expert (a stable counting sort), losses per expert in token order.
// ---------------------------------------------------------------------------
constexpr int kSmallThreads = 512;
constexpr int kStageBytes = 96 * 1024;  // LDS for the staged router and token rows (gfx950: 160 KiB per workgroup)
// LDS of the routing code behind the staging area: prob, lsev, sexp, cnt, off, aux_term (see route_small_body)
constexpr int kRouteFixedBytes = (kSmallRouteMaxPairs + kSmallRouteMaxTokens + kSmallRouteMaxTokens * kMaxTopK +
                                  2 * (kMaxExperts + 1) + kMaxExperts) * 4 + 64;
// softmax_rows (src/moe.rs, softmax over one row) and route (src/moe.rs:553-593) of one token, by one
// thread, the row used where it lies in LDS: the path for more experts than a wave has lanes.
__device__ __forceinline__ void token_phase_serial(float* row, int t, int E, int k, const uint8_t* valid, float* P,
                                                   float* lse, float* lsev, int* sexp, int* expert_of, float* gate_of) {
    const float neg_inf = __uint_as_float(0xff800000u);
    float mx = neg_inf;
    for (int e = 0; e < E; ++e)
        if (row[e] > mx) mx = row[e];  // a NaN never replaces the maximum
    float sum = 0.0f;
    for (int e = 0; e < E; ++e) {
        row[e] = rb_expf(__fadd_rn(row[e], -mx));
        sum = __fadd_rn(sum, row[e]);
    }
    const float l = __fadd_rn(mx, rb_logf(sum));
    lsev[t] = l;
    lse[t] = l;
    for (int e = 0; e < E; ++e) {
        if (sum > 0.0f) row[e] = __fdiv_rn(row[e], sum);
        P[(size_t)t * E + e] = row[e];
    }

    int* eo = sexp + t * k;
    const bool ok = (valid == nullptr) || (valid[t] != 0);
    if (!ok) {
        for (int r = 0; r < k; ++r) {
            eo[r] = -1;
            expert_of[t * k + r] = -1;
            gate_of[t * k + r] = 0.0f;
        }
        return;
    }
    float total = 0.0f;
    for (int r = 0; r < k; ++r) {
        int best = -1;
        float bestv = 0.0f;
        for (int e = 0; e < E; ++e) {
            bool taken = false;
            for (int q = 0; q < r; ++q) taken = taken || (eo[q] == e);
            if (taken) continue;
            const float v = row[e];
            if (best < 0 || v > bestv) {
                best = e;
                bestv = v;
            }
        }
        eo[r] = best;
        total = __fadd_rn(total, bestv);
        gate_of[t * k + r] = bestv;  // rewritten below once the sum is known
        expert_of[t * k + r] = best;
    }
    if (total > 0.0f)
        for (int r = 0; r < k; ++r) gate_of[t * k + r] = __fdiv_rn(row[eo[r]], total);
}

// The same two steps with G lanes per token (G = 16 or 64, E <= G), lane j holding expert j: the
// exponentials, divisions and the argmax of every round run side by side, and only what the reference
// does in sequence stays a sequence - the sum of the exponentials in index order (every lane of the group
// adds the E values up in the same order, fetching them with shuffles) and the running sum of the selected
// probabilities.  A round's winner is the largest 64-bit key (probability bits above the inverted index:
// probabilities are >= +0, so their bit patterns order like their values, and among equal ones the lower
// index wins, as the reference's strict `>` scan does); a taken expert's key is 0, and so is a NaN's, which the
// scan never prefers to anything and never replaces once it is the candidate.
// softmax_rows and route of one token by a group of G lanes (16 or 64), lane j owning expert j: the reductions
// run through lane-permuting operands (group_reduce) and the ordered sum as a lane-shift chain, so the phase makes two trips to LDS
// instead of dozens.  The chain: in every step a lane takes the sum of the lane below (a shift of the whole wave by one lane inside
// the add) and adds its own exponential, a group's first lane keeps its own, so that after l steps lane l holds ((ex_0 + ex_1) + ...)
// + ex_l; lanes past the last expert add zeros, and the last lane's sum is the token's.
template <int G>
__device__ __forceinline__ void token_phase_lanes(float* row_lds, int t, int j, int E, int k, const uint8_t* valid,
                                                  float* P, float* lse, float* lsev, int* sexp, int* expert_of,
                                                  float* gate_of) {
    const int lane = threadIdx.x & 63;
    const int base = lane - j;  // first lane of the group
    const bool mine = j < E;
    const float neg_inf = __uint_as_float(0xff800000u);
    const float v = mine ? row_lds[j] : neg_inf;
    const float mx = group_fmax((v == v) ? v : neg_inf, G);  // a NaN never replaces the maximum
    const float ex = mine ? rb_expf(__fadd_rn(v, -mx)) : 0.0f;   // lanes without an expert carry +0 through the sum
    // ((ex_0 + ex_1) + ex_2) + ...: lane l holds the sum through expert l after l steps
    float acc = ex;
    for (int st = 1; st < G; ++st) {
        const float below = __uint_as_float(lanes_from<0x138>(__float_as_uint(acc)));  // wave_shr:1
        const float next = __fadd_rn(below, ex);
        acc = j == 0 ? ex : next;
    }
    const float sum = __shfl(acc, base + G - 1);
    const float l = __fadd_rn(mx, rb_logf(sum));
    const float p = sum > 0.0f ? __fdiv_rn(ex, sum) : ex;
    if (mine) {
        P[(size_t)t * E + j] = p;
        row_lds[j] = p;  // the loss phase reads the probabilities from LDS
    }
    if (j == 0) {
        lsev[t] = l;
        lse[t] = l;
    }
    const bool ok = (valid == nullptr) || (valid[t] != 0);
    if (!ok) {
        if (j < k) {
            sexp[t * k + j] = -1;
            expert_of[t * k + j] = -1;
            gate_of[t * k + j] = 0.0f;
        }
        return;
    }
    // A NaN is never greater than anything and nothing is greater than a NaN (src/moe.rs:566-581): a NaN takes
    // part in no comparison - it is selected only when it is the first expert not yet taken, and then nothing
    // replaces it.
    const bool is_nan = p != p;
    bool taken = !mine;
    const unsigned long long gmask = G == 64 ? ~0ull : ((1ull << G) - 1ull);
    float total = 0.0f;
    float my_p = 0.0f;  // lane r keeps round r's probability
    int my_e = -1;
    for (int r = 0; r < k; ++r) {
        // greatest probability bits among the experts not yet taken (probabilities are never negative), then the
        // lowest index among the lanes that hold them
        const bool cand = !taken && !is_nan;
        const uint32_t mbits = group_umax(cand ? __float_as_uint(p) : 0u, G);
        const uint32_t ci = group_umin((cand && __float_as_uint(p) == mbits) ? (uint32_t)j : 0x7fffffffu, G);
        const unsigned long long untaken = (__ballot(!taken) >> base) & gmask;
        const unsigned long long nans = (__ballot(!taken && is_nan) >> base) & gmask;
        const int first = __ffsll((long long)untaken) - 1;  // k <= E: some expert is always left
        const bool first_nan = ((nans >> first) & 1ull) != 0ull;
        const bool use_first = first_nan || ci == 0x7fffffffu;
        const int be = use_first ? first : (int)ci;
        float bv = __uint_as_float(mbits);  // the winner's probability is the greatest bits themselves
        if (__ballot(use_first) != 0ull) {  // uniform over the wave: only a NaN first expert has to be fetched
            const float fv = __shfl(p, base + be);
            if (use_first) bv = fv;
        }
        total = __fadd_rn(total, bv);
        if (j == be) taken = true;
        if (j == r) {
            my_p = bv;
            my_e = be;
        }
    }
    if (j < k) {
        sexp[t * k + j] = my_e;
        expert_of[t * k + j] = my_e;
        gate_of[t * k + j] = total > 0.0f ? __fdiv_rn(my_p, total) : my_p;
    }
}

// What a routed call leaves for its consumers (see Work).
struct SmallTables {
    int *counts, *offsets, *tile_expert, *tile_row0, *tile_rows, *ntiles;
    float* losses;
    int *perm_slot, *perm_token, *inv_pos;
};

// The bucket loop and the losses of a call of at most 32 tokens, by one workgroup of kSmallThreads: `prob` [T, E]
// probabilities, `lsev` [T], `sexp` [T k] experts of the slots (-1: none), all in LDS and met at a barrier; `cnt`, `off`
// [kMaxExperts + 1] and `aux_term` [kMaxExperts]: scratch in LDS.
__device__ __forceinline__ void small_layout(const float* __restrict__ prob, const float* __restrict__ lsev, const int* __restrict__ sexp,
                                             int* __restrict__ cnt, int* __restrict__ off, float* __restrict__ aux_term,
                                             const uint8_t* __restrict__ valid, int T, int E, int k, float w_aux, float w_z,
                                             int tile_m, const SmallTables& o) {
    int* __restrict__ const counts = o.counts;
    int* __restrict__ const offsets = o.offsets;
    int* __restrict__ const tile_expert = o.tile_expert;
    int* __restrict__ const tile_row0 = o.tile_row0;
    int* __restrict__ const tile_rows = o.tile_rows;
    int* __restrict__ const ntiles = o.ntiles;
    float* __restrict__ const losses = o.losses;
    int* __restrict__ const perm_slot = o.perm_slot;
    int* __restrict__ const perm_token = o.perm_token;
    int* __restrict__ const inv_pos = o.inv_pos;
    const int tid = threadIdx.x;
    const int S = T * k;
    // ---- bucket loop: a stable counting sort of the slots by expert ----------------
    // With at most 64 slots and 64 experts the first wave sorts and the second wave works out the two losses beside
    // it (same formulas and orders as the general code at the end; the per-expert counts it needs are ballots of
    // its own), and nothing is left to wait for.
    const bool side_losses = S <= 64 && E <= 64;
    if (side_losses && tid >= 64 && tid < 128) {
        const int ln = tid - 64;
        const int my = ln < S ? sexp[ln] : -1;
        int c_mine = 0;  // lane e: slots of expert e
        for (int e = 0; e < E; ++e) {
            const int c = __popcll(__ballot(my == e));
            if (ln == e) c_mine = c;
        }
        int V = 0;
        for (int t = 0; t < T; ++t) V += ((valid == nullptr) || valid[t]) ? 1 : 0;
        if (ln < E) {
            float term = 0.0f;
            if (V > 0) {
                const float load = (float)c_mine / ((float)V * (float)k);
                float mass = 0.0f;
                for (int t = 0; t < T; ++t)
                    if ((valid == nullptr) || valid[t]) mass = mass + prob[t * E + ln];
                mass = mass / (float)V;
                term = load * mass;
            }
            aux_term[ln] = term;
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's LDS writes have landed
        __builtin_amdgcn_wave_barrier();
        if (ln == 0) {
            float aux = 0.0f, z = 0.0f;
            if (V > 0) {
                for (int e = 0; e < E; ++e) aux = aux + aux_term[e];
                aux = aux * ((float)E * w_aux);
                float zs = 0.0f;
                for (int t = 0; t < T; ++t)
                    if ((valid == nullptr) || valid[t]) zs = zs + lsev[t] * lsev[t];
                z = w_z * zs / (float)V;
            }
            losses[0] = aux;
            losses[1] = z;
        }
    }
    if (S <= 64) {
        // one wave, slot = lane: a ballot per expert gives its count and every slot's rank
        if (tid < 64) {
            const int my = tid < S ? sexp[tid] : -1;
            int run = 0, tiles = 0;
            if (E <= 64) {
                // the loop keeps everything in registers - slot `tid` its position, lane e expert e's count, first
                // position and first tile - and every store follows it, side by side
                int pos = -1, e_cnt = 0, e_off = 0, e_tile0 = 0;
                for (int e = 0; e < E; ++e) {
                    const unsigned long long mask = __ballot(my == e);
                    const int c = __popcll(mask);
                    pos = my == e ? run + __popcll(mask & ((1ull << tid) - 1ull)) : pos;
                    e_cnt = tid == e ? c : e_cnt;
                    e_off = tid == e ? run : e_off;
                    e_tile0 = tid == e ? tiles : e_tile0;
                    run += c;
                    tiles += c <= tile_m ? (c > 0 ? 1 : 0) : (c + tile_m - 1) / tile_m;
                }
                if (my >= 0) {
                    perm_slot[pos] = tid;
                    perm_token[pos] = tid / k;
                    inv_pos[tid] = pos;
                }
                if (tid < E) {
                    cnt[tid] = e_cnt;
                    counts[tid] = e_cnt;
                    offsets[tid] = e_off;
                    for (int r0 = 0, ti = e_tile0; r0 < e_cnt; r0 += tile_m, ++ti) {
                        tile_expert[ti] = tid;
                        tile_row0[ti] = e_off + r0;
                        tile_rows[ti] = min(tile_m, e_cnt - r0);
                    }
                }
            } else
            for (int e = 0; e < E; ++e) {
                const unsigned long long mask = __ballot(my == e);
                const int c = __popcll(mask);
                if (my == e) {
                    const int pos = run + __popcll(mask & ((1ull << tid) - 1ull));
                    perm_slot[pos] = tid;
                    perm_token[pos] = tid / k;
                    inv_pos[tid] = pos;
                }
                if (tid == 0) {
                    cnt[e] = c;
                    counts[e] = c;
                    offsets[e] = run;
                    for (int r0 = 0; r0 < c; r0 += tile_m) {
                        tile_expert[tiles] = e;
                        tile_row0[tiles] = run + r0;
                        tile_rows[tiles] = min(tile_m, c - r0);
                        ++tiles;
                    }
                }
                run += c;
            }
            if (tid < S && my < 0) inv_pos[tid] = -1;
            if (tid == 0) {
                offsets[E] = run;
                ntiles[0] = tiles;
            }
        }
    } else {
        // one expert per thread, slots in increasing order
        for (int e = tid; e < E; e += kSmallThreads) {
            int c = 0;
            for (int s = 0; s < S; ++s) c += (sexp[s] == e) ? 1 : 0;
            cnt[e] = c;
        }
        __syncthreads();
        if (tid == 0) {
            int run = 0, tiles = 0;
            for (int e = 0; e < E; ++e) {
                off[e] = run;
                counts[e] = cnt[e];
                offsets[e] = run;
                for (int r0 = 0; r0 < cnt[e]; r0 += tile_m) {
                    tile_expert[tiles] = e;
                    tile_row0[tiles] = run + r0;
                    tile_rows[tiles] = min(tile_m, cnt[e] - r0);
                    ++tiles;
                }
                run += cnt[e];
            }
            off[E] = run;
            offsets[E] = run;
            ntiles[0] = tiles;
        }
        for (int s = tid; s < S; s += kSmallThreads)
            if (sexp[s] < 0) inv_pos[s] = -1;
        __syncthreads();
        for (int e = tid; e < E; e += kSmallThreads) {
            int pos = off[e];
            for (int s = 0; s < S; ++s)
                if (sexp[s] == e) {
                    perm_slot[pos] = s;
                    perm_token[pos] = s / k;
                    inv_pos[s] = pos;
                    ++pos;
                }
        }
    }
    if (side_losses) return;
    __syncthreads();

    // ---- auxiliary losses (src/moe.rs:325-337): per expert in token order ---------
    int V = 0;
    for (int t = 0; t < T; ++t) V += ((valid == nullptr) || valid[t]) ? 1 : 0;
    for (int e = tid; e < E; e += kSmallThreads) {
        float term = 0.0f;
        if (V > 0) {
            const float load = (float)cnt[e] / ((float)V * (float)k);
            float mass = 0.0f;
            for (int t = 0; t < T; ++t)
                if ((valid == nullptr) || valid[t]) mass = mass + prob[t * E + e];
            mass = mass / (float)V;
            term = load * mass;
        }
        aux_term[e] = term;
    }
    __syncthreads();
    if (tid == 0) {
        float aux = 0.0f, z = 0.0f;
        if (V > 0) {
            for (int e = 0; e < E; ++e) aux = aux + aux_term[e];
            aux = aux * ((float)E * w_aux);
            float zs = 0.0f;
            for (int t = 0; t < T; ++t)
                if ((valid == nullptr) || valid[t]) zs = zs + lsev[t] * lsev[t];
            z = w_z * zs / (float)V;
        }
        losses[0] = aux;
        losses[1] = z;
    }
}

// STAGE = bytes of `smem` for the staged router and token rows; the routing arrays follow them.
template <typename XT, int STAGE>
__device__ __forceinline__ void route_small_body(
    unsigned char* __restrict__ smem,
    const XT* __restrict__ x, const float* __restrict__ wr, const float* __restrict__ bias,
    const uint8_t* __restrict__ valid, int T, int d, int E, int k, float w_aux, float w_z, int tile_m,
    float* __restrict__ P, float* __restrict__ lse, int* __restrict__ expert_of, float* __restrict__ gate_of,
    int* __restrict__ counts, int* __restrict__ offsets, int* __restrict__ tile_expert,
    int* __restrict__ tile_row0, int* __restrict__ tile_rows, int* __restrict__ ntiles,
    float* __restrict__ losses, int* __restrict__ perm_slot, int* __restrict__ perm_token,
    int* __restrict__ inv_pos, const float* __restrict__ norm_w, float norm_eps, XT* __restrict__ xn_out,
    bf16_t* __restrict__ rows16) {
    static_assert(STAGE % 16 == 0, "the arrays behind the staging area stay aligned");
    unsigned char* const stage = smem;
    float* const prob = reinterpret_cast<float*>(smem + STAGE);                 // [kSmallRouteMaxPairs]
    float* const lsev = prob + kSmallRouteMaxPairs;                             // [kSmallRouteMaxTokens]
    int* const sexp = reinterpret_cast<int*>(lsev + kSmallRouteMaxTokens);      // [kSmallRouteMaxTokens * kMaxTopK]
    int* const cnt = sexp + kSmallRouteMaxTokens * kMaxTopK;                    // [kMaxExperts + 1]
    int* const off = cnt + (kMaxExperts + 1);                                   // [kMaxExperts + 1]
    float* const aux_term = reinterpret_cast<float*>(off + (kMaxExperts + 1));  // [kMaxExperts]

    const int tid = threadIdx.x;
    const int lane = tid & 63;

    // ---- logits ---------------------------------------------------------------
    // When they fit, the router rows and the token rows are first copied to LDS with wide
    // coalesced loads (one round trip to memory instead of one per batch of columns); rows are
    // padded by 8 elements so that the eight pairs a wave works on fall into different banks.
    const int ds = d + 8;
    const bool staged = (d % 8 == 0) && ((size_t)E * ds * 4 + (size_t)T * ds * sizeof(XT) <= (size_t)STAGE) &&
                        (reinterpret_cast<uintptr_t>(x) % 16 == 0) && (reinterpret_cast<uintptr_t>(wr) % 16 == 0);
    if (staged) {
        float* ws = reinterpret_cast<float*>(stage);
        XT* xs = reinterpret_cast<XT*>(stage + (size_t)E * ds * 4);
        const int wp = d / 4, xp = d * (int)sizeof(XT) / 16;  // 16-byte pieces per row
        const int nw = E * wp, nx = T * xp;
        const uint4* wsrc = reinterpret_cast<const uint4*>(wr);
        const uint4* xsrc = reinterpret_cast<const uint4*>(x);
        // One load a piece from a chosen address (not a chosen one of two loads: loads under a branch stay in front
        // of their own stores, and the round trips follow one another), into variables of their own (an array of
        // pieces ends up in scratch memory).
        auto fetch = [&](int i) -> uint4 {
            i = min(i, nw + nx - 1);
            const uint4* const from = i < nw ? wsrc + i : xsrc + (i - nw);
            return *from;
        };
        auto put = [&](int i, const uint4& v) {
            if (i < nw) {
                const int r = i / wp, c = i - r * wp;
                *reinterpret_cast<uint4*>(ws + (size_t)r * ds + 4 * c) = v;
            } else if (i < nw + nx) {
                const int r = (i - nw) / xp, c = (i - nw) - r * xp;
                *reinterpret_cast<uint4*>(reinterpret_cast<char*>(xs + (size_t)r * ds) + 16 * c) = v;
            }
        };
        // eight pieces a thread are requested before the first is stored: 64 KB a round trip (36 KB for 8 tokens,
        // 8 experts and 768 columns: one)
        constexpr int NT = kSmallThreads;
        for (int i = tid; i < nw + nx; i += 8 * NT) {
            const uint4 v0 = fetch(i), v1 = fetch(i + NT), v2 = fetch(i + 2 * NT), v3 = fetch(i + 3 * NT);
            const uint4 v4 = fetch(i + 4 * NT), v5 = fetch(i + 5 * NT), v6 = fetch(i + 6 * NT), v7 = fetch(i + 7 * NT);
            __builtin_amdgcn_sched_barrier(0);
            put(i, v0); put(i + NT, v1); put(i + 2 * NT, v2); put(i + 3 * NT, v3);
            put(i + 4 * NT, v4); put(i + 5 * NT, v5); put(i + 6 * NT, v6); put(i + 7 * NT, v7);
        }
        __syncthreads();
        if (norm_w != nullptr) {
            // RmsNorm::forward (src/norm.rs:41-61) on the staged rows, in place: thread t adds up the squares
            // of row t in index order (the reference's sequential sum), then the block scales the rows with two
            // separately rounded products, rounds them to the activation type, and writes them out for the
            // kernels that follow.  (The launcher passes the norm only when the rows are staged.)
            float* const inv = lsev;  // free until the token phase
            constexpr int VN = Vec16<XT>::N;  // d is a multiple of 8 here, rows start on 16-byte boundaries
            if (tid < T) {
                const XT* row = xs + (size_t)tid * ds;
                float sum = 0.0f;
#pragma unroll 4
                for (int c = 0; c < d; c += VN) {
                    float v[VN];
                    Vec16<XT>::load(row + c, v);
#pragma unroll
                    for (int i = 0; i < VN; ++i) sum = __fadd_rn(sum, __fmul_rn(v[i], v[i]));
                }
                const float mean_square = __fdiv_rn(sum, (float)d);
                // correctly rounded root: in double, rounded once (the f32 root instruction is not)
                inv[tid] = __fdiv_rn(1.0f, (float)sqrt((double)__fadd_rn(mean_square, norm_eps)));
            }
            __syncthreads();
            const int pieces = d / VN;
            for (int i = tid; i < T * pieces; i += kSmallThreads) {
                const int t = i / pieces, c = (i - t * pieces) * VN;
                float v[VN], o[VN];
                Vec16<XT>::load(xs + (size_t)t * ds + c, v);
                const float sc = inv[t];
#pragma unroll
                for (int q = 0; q < VN; ++q) o[q] = __fmul_rn(__fmul_rn(v[q], sc), norm_w[c + q]);
                Vec16<XT>::store(xs + (size_t)t * ds + c, o);
                Vec16<XT>::store(xn_out + (size_t)t * d + c, o);
            }
            __syncthreads();
        }
        if constexpr (sizeof(XT) == 4) {
            // f32 rows of a layer whose expert products run on the bf16 matrix cores: their bf16 copy (nearest
            // even), from the staged - and, with a norm, normed - rows
            if (rows16 != nullptr) {
                for (int i = tid; i < T * (d / 8); i += kSmallThreads) {
                    const int t = i / (d / 8), c = (i - t * (d / 8)) * 8;
                    const float* src = reinterpret_cast<const float*>(xs) + (size_t)t * ds + c;
                    uint4 o;
                    o.x = f32_to_bf16_bits(src[0]) | ((uint32_t)f32_to_bf16_bits(src[1]) << 16);
                    o.y = f32_to_bf16_bits(src[2]) | ((uint32_t)f32_to_bf16_bits(src[3]) << 16);
                    o.z = f32_to_bf16_bits(src[4]) | ((uint32_t)f32_to_bf16_bits(src[5]) << 16);
                    o.w = f32_to_bf16_bits(src[6]) | ((uint32_t)f32_to_bf16_bits(src[7]) << 16);
                    *reinterpret_cast<uint4*>(rows16 + (size_t)t * d + c) = o;
                }
            }
        }
        const int tasks = T * E * 8;
        for (int base = 0; base < tasks; base += kSmallThreads) {
            const int task = base + tid;
            const bool live = task < tasks;
            const int pair = live ? task >> 3 : 0;
            const int j = task & 7;
            const int t = pair / E;
            const int e = pair - t * E;
            const XT* xr = xs + (size_t)t * ds;
            const float* wrow = ws + (size_t)e * ds;
            const float bv = (bias && live && j == 0) ? bias[e] : 0.0f;  // fetched while the dot product runs
            float acc = 0.0f;
            if (live) {
#pragma unroll 16
                for (int c = j; c < d; c += 8) acc = __fadd_rn(acc, __fmul_rn(to_f32(xr[c]), wrow[c]));
            }
            float sum = 0.0f;
#pragma unroll
            for (int l = 0; l < 8; ++l) sum = __fadd_rn(sum, __shfl(acc, (lane & ~7) + l));
            if (live && j == 0) {
                float v = __fadd_rn(sum, 0.0f);  // the reference adds its (empty) scalar rest: sum + 0
                if (bias) v = __fadd_rn(v, bv);
                prob[pair] = v;
            }
        }
    } else {
        const int tail = d - d % 8;
        const int tasks = T * E * 8;
        for (int base = 0; base < tasks; base += kSmallThreads) {
            const int task = base + tid;
            const bool live = task < tasks;
            const int pair = live ? task >> 3 : 0;
            const int j = task & 7;
            const int t = pair / E;
            const int e = pair - t * E;
            const XT* xr = x + (size_t)t * d;
            const float* wrow = wr + (size_t)e * d;
            // lane j of the pair: columns j, j + 8, ... in increasing order.  The loads of 32 steps
            // are issued together (they do not depend on one another); the adds stay a chain.
            float acc = 0.0f;
            if (live) {
                constexpr int U = 32;
                for (int c0 = j; c0 < tail; c0 += 8 * U) {
                    float xv[U], wv[U];
    #pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int c = c0 + 8 * u;
                        const int cc = c < tail ? c : j;  // always a valid column: no branch around the load
                        xv[u] = to_f32(xr[cc]);
                        wv[u] = wrow[cc];
                    }
    #pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (c0 + 8 * u < tail) acc = __fadd_rn(acc, __fmul_rn(xv[u], wv[u]));
                }
            }
            // lanes folded left to right, by the first thread of the group of eight
            float sum = 0.0f;
    #pragma unroll
            for (int l = 0; l < 8; ++l) sum = __fadd_rn(sum, __shfl(acc, (lane & ~7) + l));
            if (live && j == 0) {
                float rest = 0.0f;
                for (int c = tail; c < d; ++c) rest = __fadd_rn(rest, __fmul_rn(to_f32(xr[c]), wrow[c]));
                float v = __fadd_rn(sum, rest);
                if (bias) v = __fadd_rn(v, bias[e]);
                prob[pair] = v;
            }
        }
    }
    __syncthreads();

    // ---- softmax_rows and route: one token per thread --------------------------
    // Up to 64 experts: a group of lanes per token; more: one thread per token.
    if (E <= 16 && k <= 16) {
        // 16 lanes per token, 32 tokens per pass of the block
        for (int t = tid >> 4; t < T; t += kSmallThreads / 16)
            token_phase_lanes<16>(prob + t * E, t, tid & 15, E, k, valid, P, lse, lsev, sexp, expert_of, gate_of);
    } else if (E <= 64) {
        // a wave per token (k <= 32 < 64 always)
        for (int t = tid >> 6; t < T; t += kSmallThreads / 64)
            token_phase_lanes<64>(prob + t * E, t, tid & 63, E, k, valid, P, lse, lsev, sexp, expert_of, gate_of);
    } else if (tid < T) {
        token_phase_serial(prob + tid * E, tid, E, k, valid, P, lse, lsev, sexp, expert_of, gate_of);
    }
    __syncthreads();

    small_layout(prob, lsev, sexp, cnt, off, aux_term, valid, T, E, k, w_aux, w_z, tile_m,
                 SmallTables{counts, offsets, tile_expert, tile_row0, tile_rows, ntiles, losses, perm_slot, perm_token, inv_pos});
}

template <typename XT>
__global__ __launch_bounds__(kSmallThreads) void route_small_kernel(
    const XT* __restrict__ x, const float* __restrict__ wr, const float* __restrict__ bias,
    const uint8_t* __restrict__ valid, int T, int d, int E, int k, float w_aux, float w_z, int tile_m,
    float* __restrict__ P, float* __restrict__ lse, int* __restrict__ expert_of, float* __restrict__ gate_of,
    int* __restrict__ counts, int* __restrict__ offsets, int* __restrict__ tile_expert,
    int* __restrict__ tile_row0, int* __restrict__ tile_rows, int* __restrict__ ntiles,
    float* __restrict__ losses, int* __restrict__ perm_slot, int* __restrict__ perm_token,
    int* __restrict__ inv_pos, const float* __restrict__ norm_w, float norm_eps, XT* __restrict__ xn_out,
    bf16_t* __restrict__ rows16) {
    __shared__ __align__(16) unsigned char smem[kStageBytes + kRouteFixedBytes];
    route_small_body<XT, kStageBytes>(smem, x, wr, bias, valid, T, d, E, k, w_aux, w_z, tile_m, P, lse, expert_of, gate_of,
                                      counts, offsets, tile_expert, tile_row0, tile_rows, ntiles, losses, perm_slot,
                                      perm_token, inv_pos, norm_w, norm_eps, xn_out, rows16);
}

bool small_route_ok(int T, int E, int k) {
    return T >= 1 && T <= kSmallRouteMaxTokens && E <= kMaxExperts && k <= kMaxTopK &&
           T * E <= kSmallRouteMaxPairs;
}

// Whether route_small_kernel copies the router and the token rows into LDS for this call (the condition the
// kernel itself evaluates); only then can it apply the norm in front of the layer.
bool small_route_stages_rows(const void* x, const float* wr, int T, int d, int E, bool bf16) {
    const size_t ds = (size_t)d + 8;
    return d % 8 == 0 && (size_t)E * ds * 4 + (size_t)T * ds * (bf16 ? 2 : 4) <= (size_t)kStageBytes &&
           reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(wr) % 16 == 0;
}

hipError_t launch_route_small(const SmallRouteArgs& a, bool bf16, hipStream_t s) {
    if (!small_route_ok(a.T, a.E, a.k)) return hipErrorInvalidValue;
    if (a.norm_w && (!a.xn_out || !small_route_stages_rows(a.x, a.wr, a.T, a.d, a.E, bf16))) return hipErrorInvalidValue;
    if (a.rows16 && (bf16 || !small_route_stages_rows(a.x, a.wr, a.T, a.d, a.E, bf16))) return hipErrorInvalidValue;
    if (bf16)
        RB_LAUNCH(route_small_kernel<bf16_t>, dim3(1), dim3(kSmallThreads), 0, s,
                           static_cast<const bf16_t*>(a.x), a.wr, a.bias, a.valid, a.T, a.d, a.E, a.k, a.w_aux, a.w_z,
                           a.tile_m, a.P, a.lse, a.expert_of, a.gate_of, a.counts, a.offsets, a.tile_expert,
                           a.tile_row0, a.tile_rows, a.ntiles, a.losses, a.perm_slot, a.perm_token, a.inv_pos,
                           a.norm_w, a.norm_eps, static_cast<bf16_t*>(a.xn_out), nullptr);
    else
        RB_LAUNCH(route_small_kernel<float>, dim3(1), dim3(kSmallThreads), 0, s,
                           static_cast<const float*>(a.x), a.wr, a.bias, a.valid, a.T, a.d, a.E, a.k, a.w_aux, a.w_z,
                           a.tile_m, a.P, a.lse, a.expert_of, a.gate_of, a.counts, a.offsets, a.tile_expert,
                           a.tile_row0, a.tile_rows, a.ntiles, a.losses, a.perm_slot, a.perm_token, a.inv_pos,
                           a.norm_w, a.norm_eps, static_cast<float*>(a.xn_out), static_cast<bf16_t*>(a.rows16));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// decode_gemm_kernel: out[row, n] for one tile of at most 32 rows and one block of 32
// output features (gate/up: 32 gate rows and the matching 32 up rows of the packed weights).
// The waves of a workgroup take an equal share of the reduction steps each; a wave fetches
// its weight fragments (1 KB per step and row block, straight from the packed layout) in
// batches of kBatch steps so that tens of kilobytes are in flight, multiplies them on the
// matrix cores against token fragments read from global memory (32 rows x K: they stay in
// L2), and the partial sums meet in LDS, in a fixed order.
// blockIdx.y < max_tiles: routed tiles (those past *ntiles exit); the rest: 32-row blocks of
// the shared expert, which takes every token.
// ---------------------------------------------------------------------------
constexpr int kBatch = 12;

// Partial sums meet in LDS as [wave][gate, up][16][64 lanes], the rows of 64 this far apart: the threads that add them up read
// 8 neighbouring lanes of rows 0, 4, 8 and 12, which then lie in 64 different banks.  What follows the products of the int8
// front launch at 32 tokens, d 768, 8 experts of 1408: 2.7 us 64 apart, 1.5 so, the scales requested in front of the products.
constexpr int kRedPitch = 66;
struct DecodeSide {
    const bf16_t* a;
    const int* row_index;
    const char* w;
    const float* scales;
    bf16_t* out;
    int N, K, row0, rows;
    int a_row0;    // added to a row's number in `a` (rows of one expert inside a per-expert array)
    int out_row0;  // first output row is out_row0 + row0
    // The rows are read again inside this launch by a workgroup that may sit on another XCD (the folded combine): the
    // XCDs' L2 caches are not coherent with one another, so such rows are stored with device-scope stores, which
    // go through to memory, and read back with device-scope loads.
    bool coherent_out = false;
    // rows behind a norm (RowForm with kNorm), in LDS: the norm's weights [K] and the rows' factors [32]
    const float* norm_w = nullptr;
    const float* row_factor = nullptr;
    bool widen_first = false;  // int8 weights of the first batch are widened in front of the hook
};

// The rows a product reads.  XT: bf16, or f32 rounded to bf16 on the way (the product's precision either way).  NORM: the
// rows are raw and the product is taken of their normed form, value * factor * weight with the norm's own roundings
// (src/norm.rs:41-61), as if the normed rows had been written out first.
template <typename XT, bool NORM>
struct RowForm {
    typedef XT type;
    static constexpr bool kNorm = NORM;
    static constexpr bool kPlain = !NORM && sizeof(XT) == 2;
};
struct NoHook {
    __device__ __forceinline__ void operator()() const {}
};

// For a launch with one row of workgroups per EXPERT (decode_down_by_expert_kernel): which rows the expert has is read off
// the experts of the call's slots, fetched in front of the first weight loads and looked at behind them.
constexpr int kLateRounds = 4;  // 64 slots a round: at most 8 slots a token
struct LateRows {
    const int* expert_of;  // [S]
    int S, k, expert;
    int* row_slot;         // LDS [32]: the slot of every row of the side, ascending
    bool routed;           // false: the side's rows are sd.row0 / sd.rows as they stand (the shared expert)
};

template <bool SWIGLU, bool I8, int NW, int BATCH, int TEAMS = 1, bool LATE_ROWS = false, typename ROWS = RowForm<bf16_t, false>,
          typename HOOK = NoHook>
__device__ __forceinline__ void decode_gemm_body(DecodeSide& sd, int fb, float* red_raw, LateRows* late = nullptr, HOOK hook = HOOK{});

constexpr int kCombineEarlySlots = 4;  // slots a token up to which a thread fetches what the combine needs beforehand

// The combine of a decode-shaped call, for the 32 output features of block `fb` and every token: what
// combine_vec_kernel computes, element by element in the same order (the token's expert rows by ascending position,
// i.e. ascending expert; gate * row as a rounded multiply, then a rounded add; then the shared expert's row; then
// the residual).  Run by the last workgroup of the block's column to finish; the rows were stored with device-scope
// stores and are read with device-scope loads (see DecodeSide::coherent_out).
template <typename XT>
__device__ __forceinline__ void decode_combine_block(const DecodeGemmArgs& g, int fb, int nthreads) {
    const bf16_t* const y = static_cast<const bf16_t*>(g.out);
    const bf16_t* const ys = g.a_shared ? static_cast<const bf16_t*>(g.out_shared) : nullptr;
    const XT* const res = static_cast<const XT*>(g.cmb_residual);
    XT* const out = static_cast<XT*>(g.cmb_out);
    const int d = g.N, k = g.cmb_k;
    for (int idx = threadIdx.x; idx < g.cmb_T * 16; idx += nthreads) {
        const int t = idx >> 4;
        const int c = fb * 32 + 2 * (idx & 15);
        const int* const ip = g.cmb_inv_pos + (size_t)t * k;
        const float* const gp = g.cmb_gate_of + (size_t)t * k;
        float a0 = 0.0f, a1 = 0.0f;
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
            const uint32_t v = __hip_atomic_load(reinterpret_cast<const uint32_t*>(y + (size_t)best * d + c),
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const float gt = gp[bi];
            a0 = __fadd_rn(a0, __fmul_rn(gt, __uint_as_float(v << 16)));
            a1 = __fadd_rn(a1, __fmul_rn(gt, __uint_as_float(v & 0xffff0000u)));
        }
        if (ys) {
            const uint32_t v = __hip_atomic_load(reinterpret_cast<const uint32_t*>(ys + (size_t)t * d + c),
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            a0 = __fadd_rn(a0, __uint_as_float(v << 16));
            a1 = __fadd_rn(a1, __uint_as_float(v & 0xffff0000u));
        }
        if (res) {
            a0 = __fadd_rn(a0, to_f32(res[(size_t)t * d + c]));
            a1 = __fadd_rn(a1, to_f32(res[(size_t)t * d + c + 1]));
        }
        out[(size_t)t * d + c] = from_f32<XT>(a0);
        out[(size_t)t * d + c + 1] = from_f32<XT>(a1);
    }
}

// What a thread of the folded combine can fetch before its workgroup has multiplied anything: where its token's expert rows
// lie, in ascending expert order once sorted, their gates, and the residual.  BY_SLOT: the expert rows lie in slot order and
// `key` is the slot's expert; otherwise it is the row's position.  M: slots a token at most.
template <int M>
struct CombineEarly {
    int key[M];  // as the routing wrote them; slots past k repeat the last one
    float gate[M];
    uint32_t res[2];  // the residual's two elements as they lie in memory: one word of two bf16, or two f32
};

template <int M>
__device__ __forceinline__ void decode_combine_fetch(const DecodeGemmArgs& g, const int* keys, int fb, CombineEarly<M>& ce) {
    // loads only, none of them looked at here and no branch between them: they return while the weights stream in
    const int t = min((int)threadIdx.x >> 4, g.cmb_T - 1), c = fb * 32 + 2 * ((int)threadIdx.x & 15), k = g.cmb_k;
    const int* const ip = keys + (size_t)t * k;
    const float* const gp = g.cmb_gate_of + (size_t)t * k;
#pragma unroll
    for (int q = 0; q < M; ++q) {
        ce.key[q] = ip[min(q, k - 1)];
        ce.gate[q] = gp[min(q, k - 1)];
    }
    // (without a residual the words of the routing's gates are fetched and never used; bf16: the second word is the first
    // again)
    const int es = g.cmb_f32 ? 4 : 2;
    const char* const at = g.cmb_residual ? static_cast<const char*>(g.cmb_residual) + ((size_t)t * g.N + c) * es
                                          : reinterpret_cast<const char*>(g.cmb_gate_of);
    ce.res[0] = *reinterpret_cast<const uint32_t*>(at);
    ce.res[1] = *reinterpret_cast<const uint32_t*>(at + (g.cmb_f32 && g.cmb_residual ? 4 : 0));
}

// decode_combine_block for a workgroup of 512 threads (one element pair a thread) that fetched `ce` beforehand: the
// expert rows' loads go out side by side, the sums are taken in the same order.
template <typename XT, bool BY_SLOT, int M>
__device__ __forceinline__ void decode_combine_block_early(const DecodeGemmArgs& g, int fb, CombineEarly<M> ce) {
    const int t = (int)threadIdx.x >> 4, c = fb * 32 + 2 * ((int)threadIdx.x & 15);
    if (t >= g.cmb_T) return;
    // ascending keys (they are distinct; a padding token's slots and the slots past k have no row), each with its row
    int row[M];
#pragma unroll
    for (int q = 0; q < M; ++q) {
        row[q] = BY_SLOT ? t * g.cmb_k + q : ce.key[q];
        if (q >= g.cmb_k || ce.key[q] < 0) ce.key[q] = 0x7fffffff;
    }
    auto order = [&](int a, int b) {
        if (ce.key[b] < ce.key[a]) {
            const int p = ce.key[a]; ce.key[a] = ce.key[b]; ce.key[b] = p;
            const int r = row[a]; row[a] = row[b]; row[b] = r;
            const float w = ce.gate[a]; ce.gate[a] = ce.gate[b]; ce.gate[b] = w;
        }
    };
    // (neighbours exchanged in M rounds, every other pair at a time)
#pragma unroll
    for (int round = 0; round < M; ++round)
#pragma unroll
        for (int q = round & 1; q + 1 < M; q += 2) order(q, q + 1);
    const bf16_t* const y = static_cast<const bf16_t*>(g.out);
    const int d = g.N;
    uint32_t v[M], vs = 0u;
#pragma unroll
    for (int q = 0; q < M; ++q)
        v[q] = ce.key[q] != 0x7fffffff
                   ? __hip_atomic_load(reinterpret_cast<const uint32_t*>(y + (size_t)row[q] * d + c), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT)
                   : 0u;
    if (g.a_shared)
        vs = __hip_atomic_load(reinterpret_cast<const uint32_t*>(static_cast<const bf16_t*>(g.out_shared) + (size_t)t * d + c),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
    for (int q = 0; q < M; ++q)
        if (ce.key[q] != 0x7fffffff) {
            a0 = __fadd_rn(a0, __fmul_rn(ce.gate[q], __uint_as_float(v[q] << 16)));
            a1 = __fadd_rn(a1, __fmul_rn(ce.gate[q], __uint_as_float(v[q] & 0xffff0000u)));
        }
    if (g.a_shared) {
        a0 = __fadd_rn(a0, __uint_as_float(vs << 16));
        a1 = __fadd_rn(a1, __uint_as_float(vs & 0xffff0000u));
    }
    if (g.cmb_residual) {
        if constexpr (sizeof(XT) == 4) {
            a0 = __fadd_rn(a0, __uint_as_float(ce.res[0]));
            a1 = __fadd_rn(a1, __uint_as_float(ce.res[1]));
        } else {
            a0 = __fadd_rn(a0, __uint_as_float(ce.res[0] << 16));
            a1 = __fadd_rn(a1, __uint_as_float(ce.res[0] & 0xffff0000u));
        }
    }
    XT* const out = static_cast<XT*>(g.cmb_out);
    out[(size_t)t * d + c] = from_f32<XT>(a0);
    out[(size_t)t * d + c + 1] = from_f32<XT>(a1);
}

template <bool SWIGLU, bool I8, int NW>
__global__ __launch_bounds__(NW * 64) void decode_gemm_kernel(DecodeGemmArgs g) {
    __shared__ float red[NW * (SWIGLU ? 2 : 1) * 16 * kRedPitch];
    __shared__ int last_of_block;
    const int fb = blockIdx.x;
    const int ty = blockIdx.y;
    DecodeSide sd;
    sd.a_row0 = 0;
    sd.out_row0 = 0;
    // One round trip for the whole tile table: the four entries are fetched side by side (a stale entry past
    // *ntiles is read and dropped), not one after the other - with cold caches every dependent scalar load in
    // front of the first weight load is a few hundred nanoseconds of a launch that lasts ten microseconds.
    const bool routed = ty < g.max_tiles;
    const int tix = routed ? ty : 0;
    const int live_tiles = *g.ntiles;
    const int t_expert = g.tile_expert[tix], t_row0 = g.tile_row0[tix], t_rows = g.tile_rows[tix];
    asm volatile("" ::"s"(live_tiles), "s"(t_expert), "s"(t_row0), "s"(t_rows));  // all four here, not sunk into the branches
    // workgroups that write rows of this feature block's columns: the live routed tiles and the shared expert's
    const int writers = live_tiles + (g.a_shared ? (g.T_shared + 31) / 32 : 0);
    bool works = true;
    if (routed) {
        if (ty >= live_tiles) works = false;
        const int expert = t_expert;
        sd.a = static_cast<const bf16_t*>(g.a);
        sd.row_index = g.row_index;
        sd.w = static_cast<const char*>(g.w) + (size_t)expert * g.w_expert_stride * (I8 ? 1 : 2);
        sd.scales = I8 ? g.scales + (size_t)expert * g.s_expert_stride : nullptr;
        sd.out = static_cast<bf16_t*>(g.out);
        sd.N = g.N;
        sd.K = g.K;
        sd.row0 = t_row0;
        sd.rows = t_rows;
        sd.a_row0 = expert * g.a_expert_rows;
    } else {
        const int st = ty - g.max_tiles;
        sd.a = static_cast<const bf16_t*>(g.a_shared);
        sd.row_index = nullptr;
        sd.w = static_cast<const char*>(g.w_shared);
        sd.scales = I8 ? g.scales_shared : nullptr;
        sd.out = static_cast<bf16_t*>(g.out_shared);
        sd.N = g.N_shared;
        sd.K = g.K_shared;
        sd.row0 = st * 32;
        sd.rows = min(32, g.T_shared - sd.row0);
    }
    if (fb * 32 >= sd.N) return;
    if constexpr (!SWIGLU) {
        if (g.cmb_out != nullptr) {  // uniform over the launch
            // eight waves and at most four slots a token: what the combine needs of the routing is fetched now
            const bool early = NW == 8 && g.cmb_k <= kCombineEarlySlots;
            CombineEarly<kCombineEarlySlots> ce;
            if (early) decode_combine_fetch(g, g.cmb_inv_pos, fb, ce);
            if (!works) {
                // nothing to multiply here; with no writer at all (every row is padding and there is no shared
                // expert) the first of these workgroups still owes the block its combine
                if (writers != 0 || ty != 0) return;
            } else {
                sd.coherent_out = true;
                decode_gemm_body<SWIGLU, I8, NW, kBatch>(sd, fb, red);
                // every wave waits until its row stores have been acknowledged (they are device-scope stores: they
                // go through to memory) before the workgroup's arrival is counted behind the barrier - a barrier
                // alone does not wait for stores.  No device-scope fence: that would write back this XCD's whole
                // L2, once per workgroup.
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                if (threadIdx.x == 0) {
                    const int before = atomicAdd(&g.cmb_counter[fb * kDecodeCombineCounterStride], 1);
                    last_of_block = before == writers - 1;
                    if (before == writers - 1) atomicExch(&g.cmb_counter[fb * kDecodeCombineCounterStride], 0);  // every writer has arrived: ready for the next launch
                }
                __syncthreads();
                if (!last_of_block) return;
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            }
            if (early) {
                if (g.cmb_f32) decode_combine_block_early<float, false>(g, fb, ce);
                else decode_combine_block_early<bf16_t, false>(g, fb, ce);
            } else {
                if (g.cmb_f32) decode_combine_block<float>(g, fb, NW * 64);
                else decode_combine_block<bf16_t>(g, fb, NW * 64);
            }
            return;
        }
    }
    if (!works) return;
    decode_gemm_body<SWIGLU, I8, NW, kBatch>(sd, fb, red);
}

// ---------------------------------------------------------------------------
// decode_down_by_expert_kernel: the down product and the folded combine behind decode_front_kernel, blockIdx.y =
// expert (then the shared expert's 32-row blocks, then one workgroup for the tables).  decode_gemm_kernel learns its
// expert from the tile table and its rows from the row index - two dependent trips to memory in front of the weight
// loads and the token loads; here the weights' address follows from the grid, and which rows the expert has is read off
// the slots' experts, requested before the weights and looked at behind them.  Nothing of the launch waits for the
// counting sort: expert rows are stored by slot and summed by slot, in ascending expert order, and the tables that
// callers may ask for (and the losses) are made by a workgroup of their own beside the products.  Every thread also
// fetches what the combine will need of the routing before the product, so that the last workgroup of a block has only
// the expert rows left to load.  An expert without rows costs its weights' bytes.
// Same products, same order of sums: the outputs are decode_gemm_kernel's bit for bit.
// ---------------------------------------------------------------------------
constexpr int kLayoutLdsFloats = kSmallRouteMaxPairs + kSmallRouteMaxTokens + kSmallRouteMaxTokens * kMaxTopK + 2 * (kMaxExperts + 1) +
                                 kMaxExperts;

// The tables of a call whose probabilities, log-sum-exps and experts lie in memory.
__device__ __forceinline__ void layout_from_memory(float* lds, const DecodeLayoutArgs& a) {
    float* const prob = lds;
    float* const lsev = prob + kSmallRouteMaxPairs;
    int* const sexp = reinterpret_cast<int*>(lsev + kSmallRouteMaxTokens);
    int* const cnt = sexp + kSmallRouteMaxTokens * kMaxTopK;
    int* const off = cnt + (kMaxExperts + 1);
    float* const aux_term = reinterpret_cast<float*>(off + (kMaxExperts + 1));
    for (int i = threadIdx.x; i < a.T * a.E; i += kSmallThreads) prob[i] = a.P[i];
    for (int i = threadIdx.x; i < a.T * a.k; i += kSmallThreads) sexp[i] = a.expert_of[i];
    for (int i = threadIdx.x; i < a.T; i += kSmallThreads) lsev[i] = a.lse[i];
    __syncthreads();
    small_layout(prob, lsev, sexp, cnt, off, aux_term, a.valid, a.T, a.E, a.k, a.w_aux, a.w_z, kDecodeTileM,
                 SmallTables{a.counts, a.offsets, a.tile_expert, a.tile_row0, a.tile_rows, a.ntiles, a.losses, a.perm_slot,
                             a.perm_token, a.inv_pos});
}

// ... in a launch of its own, for a caller that takes the tile-table launch behind decode_front_kernel
__global__ __launch_bounds__(kSmallThreads) void decode_layout_kernel(DecodeLayoutArgs a) {
    __shared__ float lds[kLayoutLdsFloats];
    layout_from_memory(lds, a);
}

template <bool I8, int M>
__global__ __launch_bounds__(512) void decode_down_by_expert_kernel(DecodeGemmArgs g, DecodeLayoutArgs t) {
    constexpr int kRed = 8 * 16 * kRedPitch;
    __shared__ float red[kRed > kLayoutLdsFloats ? kRed : kLayoutLdsFloats];
    __shared__ int row_slot[32];
    __shared__ int last_of_block;
    const int E = t.E;
    const int fb = blockIdx.x, side = blockIdx.y;
    const int shared_tiles = g.a_shared ? (g.T_shared + 31) / 32 : 0;
    const bool routed = side < E;
    if (side == E + shared_tiles) {
        if (fb == 0) layout_from_memory(red, t);
        return;
    }
    LateRows late;
    late.routed = routed;
    late.expert_of = t.expert_of;
    late.S = t.T * t.k;
    late.k = t.k;
    late.expert = side;
    late.row_slot = row_slot;
    DecodeSide sd;
    sd.row_index = nullptr;
    sd.a_row0 = 0;
    sd.out_row0 = 0;
    sd.row0 = 0;
    sd.rows = 0;
    sd.coherent_out = true;
    if (routed) {
        sd.a = static_cast<const bf16_t*>(g.a);
        sd.a_row0 = side * g.a_expert_rows;
        sd.w = static_cast<const char*>(g.w) + (size_t)side * g.w_expert_stride * (I8 ? 1 : 2);
        sd.scales = I8 ? g.scales + (size_t)side * g.s_expert_stride : nullptr;
        sd.out = static_cast<bf16_t*>(g.out);
        sd.N = g.N;
        sd.K = g.K;
    } else {
        const int st = side - E;
        sd.a = static_cast<const bf16_t*>(g.a_shared);
        sd.w = static_cast<const char*>(g.w_shared);
        sd.scales = I8 ? g.scales_shared : nullptr;
        sd.out = static_cast<bf16_t*>(g.out_shared);
        sd.N = g.N_shared;
        sd.K = g.K_shared;
        sd.row0 = st * 32;
        sd.rows = min(32, g.T_shared - sd.row0);
    }
    CombineEarly<M> ce;
    decode_combine_fetch(g, t.expert_of, fb, ce);
    decode_gemm_body<false, I8, 8, kBatch, 1, true>(sd, fb, red, &late);
    // every side of the block arrives, with rows or without
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the row stores have been acknowledged
    __syncthreads();
    if (threadIdx.x == 0) {
        const int writers = E + shared_tiles;
        const int before = atomicAdd(&g.cmb_counter[fb * kDecodeCombineCounterStride], 1);
        last_of_block = before == writers - 1;
        if (before == writers - 1) atomicExch(&g.cmb_counter[fb * kDecodeCombineCounterStride], 0);  // every writer has arrived: ready for the next launch
    }
    __syncthreads();
    if (!last_of_block) return;
    if (g.cmb_f32) decode_combine_block_early<float, true>(g, fb, ce);
    else decode_combine_block_early<bf16_t, true>(g, fb, ce);
}

// ---------------------------------------------------------------------------
// decode_down_few_kernel: the down product and the combine of a call of a row or two, without a hand-over between workgroups.
// A workgroup owns 8 output features and takes every PAIR of a row and a side of it (a slot's expert, or the shared expert), up
// to four: a 32 x 32 x 16 multiply holds them all, 8 weight rows and one hidden row each (rows 8 j .. 8 j + 7 of one operand,
// column j of the other; the products of different pairs are dropped), so that a wave fetches whole kilobytes.  The waves
// split the reduction as in decode_gemm_body and their sums meet in LDS in the same order, so the rows are those of
// the other down launches bit for bit; the wave that adds them up has all of a token's rows and sums it on the spot.  Expert rows
// are stored for who asks for them and not waited for.
// Bound by its chain: the slots' experts, then weights and hidden rows side by side, then the sums.  decode_down_by_expert_kernel
// requests an expert's weights at once, but its rows go to memory, are counted in and come back to be summed, which takes longer
// than the one trip; and here nothing is fetched of experts without rows.  us a call, before / now: one row of the default model
// 12.25 / 11.2, without the norm 11.1 / 10.1; d 768, 8 experts of 1408, two rows 14.9 / 13.65, one row with a shared expert 15.9 /
// 14.1; int8, d 1024, two rows 16.1 / 15.5.  Behind route_small_kernel 25.4 / 24.8 (one row, 16 experts).
// A wave requests all its steps at once, up to eleven: BATCH is 3, 6 or 11, and a wave of fewer asks for its last step over and over (two
// of six times at 512 columns, three of eleven at 1024).  Far too many cost more than they save: with room for 12 where there are 3,
// one row of the default model took 12.4.
// ---------------------------------------------------------------------------
constexpr int kFewPairs = 4;  // pairs of a call at most

template <bool I8, int BATCH>
__global__ __launch_bounds__(512) void decode_down_few_kernel(DecodeGemmArgs g, DecodeLayoutArgs t) {
    constexpr int M = kFewPairs, kRed = 8 * M * 8;
    __shared__ __align__(16) float red[kRed > kLayoutLdsFloats ? kRed : kLayoutLdsFloats];
    const int blk = blockIdx.x;
    if (blk == g.N / 8) return layout_from_memory(red, t);  // (behind decode_front_kernel)
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T = t.T, k = t.k, S = T * k, P = S + (g.a_shared ? T : 0);
    const bool front = g.a_expert_rows != 0;  // hidden rows per expert and expert rows by slot, or both by position

    // ---- the pairs of this lane's operands: 8 weight rows of one, the hidden row of one
    const int a_pair = (lane & 31) >> 3, b_pair = min(lane & 31, M - 1);
    const int a_expert = t.expert_of[min(a_pair, S - 1)], b_expert = t.expert_of[min(b_pair, S - 1)];
    const int b_pos = front ? 0 : t.inv_pos[min(b_pair, S - 1)];
    // what this thread will finish: pair and feature, and as token and feature
    const int f = tid & 7, n = blk * 8 + f, pair = min(tid >> 3, P - 1), token = min(tid >> 3, T - 1);
    const int my_expert = t.expert_of[min(pair, S - 1)], my_pos = front ? pair : t.inv_pos[min(pair, S - 1)];
    int key[M], slot[M];
    float gate[M];
#pragma unroll
    for (int q = 0; q < M; ++q) {
        key[q] = t.expert_of[token * k + min(q, k - 1)];
        gate[q] = g.cmb_gate_of[token * k + min(q, k - 1)];
    }
    float residual = 0.0f;
    if (g.cmb_residual)  // uniform
        residual = g.cmb_f32 ? static_cast<const float*>(g.cmb_residual)[(size_t)token * g.N + n]
                             : to_f32(static_cast<const bf16_t*>(g.cmb_residual)[(size_t)token * g.N + n]);
    float scale_shared = 1.0f;
    if (I8 && g.a_shared) scale_shared = g.scales_shared[n];

    struct Share {  // this wave's steps of a reduction
        int first, count, last;
    };
    auto share = [&](int K) {
        const int steps = K / 16, chunk = (steps + 7) / 8;
        Share s;
        s.first = min(steps - 1, wave * chunk);  // (a wave without a step: a valid one, not used)
        s.count = min(chunk, max(steps - wave * chunk, 0));
        s.last = s.first + max(s.count - 1, 0);
        return s;
    };
    const Share sr = share(g.K), ss = g.a_shared ? share(g.K_shared) : sr;
    const int most = max(sr.count, ss.count), least = min(sr.count, ss.count);
    const bool ra = a_pair < S || !g.a_shared, rb = b_pair < S || !g.a_shared;
    const Share sa = ra ? sr : ss, sb = rb ? sr : ss;
    const char* const wa = (ra ? static_cast<const char*>(g.w) + (size_t)max(a_expert, 0) * g.w_expert_stride * (I8 ? 1 : 2)
                               : static_cast<const char*>(g.w_shared)) +
                           (size_t)(blk >> 2) * (ra ? g.K : g.K_shared) * 32 * (I8 ? 1 : 2) + (half * 32 + (blk & 3) * 8 + (lane & 7)) * 16;
    const int p = min(b_pair, P - 1);
    const int row = front ? max(b_expert, 0) * T + p / k : max(b_pos, 0);
    const bf16_t* const xb = (rb ? static_cast<const bf16_t*>(g.a) + (size_t)row * g.K
                                 : static_cast<const bf16_t*>(g.a_shared) + (size_t)(p - S) * g.K_shared) + 8 * half;
    floatx16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    // (a step past a pair's share: a valid address, and zeros in its place)
    auto batch = [&](const int u0) {
        uint4 w[BATCH], x[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            x[u] = *reinterpret_cast<const uint4*>(xb + 16 * min(sb.first + u0 + u, sb.last));
            const int s = min(sa.first + u0 + u, sa.last);
            if constexpr (I8) {
                const uint2 v = *reinterpret_cast<const uint2*>(wa + (size_t)(s >> 1) * 1024 + (s & 1) * 8);
                w[u].x = v.x;
                w[u].y = v.y;
            } else {
                w[u] = *reinterpret_cast<const uint4*>(wa + (size_t)s * 1024);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            if (u0 + u >= most) break;  // uniform
            bf16x8 wv, xv = __builtin_bit_cast(bf16x8, x[u]);
            if constexpr (I8) wv = widen_i8(make_uint2(w[u].x, w[u].y));
            else wv = __builtin_bit_cast(bf16x8, w[u]);
            if (u0 + u >= least) {  // uniform
                const bf16x8 zero = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
                if (u0 + u >= sa.count) wv = zero;
                if (u0 + u >= sb.count) xv = zero;
            }
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, xv, acc, 0, 0, 0);
        }
    };
    batch(0);
    for (int u0 = BATCH; u0 < most; u0 += BATCH) batch(u0);
    // accumulator element v of lane l: weight row 8 (v / 4) + 4 (l / 32) + v % 4, hidden row l % 32
    const int j = lane & 31;
    if (j < M) {
        float y[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) y[m] = j == 0 ? acc[m] : j == 1 ? acc[4 + m] : j == 2 ? acc[8 + m] : acc[12 + m];
        *reinterpret_cast<float4*>(red + (wave * M + j) * 8 + 4 * half) = make_float4(y[0], y[1], y[2], y[3]);
    }
    // ascending experts; a padding token's slots and the slots past k have no row
#pragma unroll
    for (int q = 0; q < M; ++q) {
        slot[q] = token * k + q;
        if (q >= k || key[q] < 0) key[q] = 0x7fffffff;
    }
#pragma unroll
    for (int round = 0; round < M; ++round)
#pragma unroll
        for (int q = round & 1; q + 1 < M; q += 2)
            if (key[q + 1] < key[q]) {
                const int a = key[q]; key[q] = key[q + 1]; key[q + 1] = a;
                const int b = slot[q]; slot[q] = slot[q + 1]; slot[q + 1] = b;
                const float c = gate[q]; gate[q] = gate[q + 1]; gate[q + 1] = c;
            }
    const bool routed = pair < S;
    float scale = scale_shared;
    if (I8 && wave == 0 && routed) scale = g.scales[(size_t)max(my_expert, 0) * g.s_expert_stride + n];
    __syncthreads();
    if (wave != 0) return;
    float y = red[pair * 8 + f];
#pragma unroll
    for (int w = 1; w < 8; ++w) y += red[(w * M + pair) * 8 + f];
    if constexpr (I8) y *= scale;
    const uint32_t bits = f32_to_bf16_bits(y);
    if (tid < 8 * P && (!routed || my_expert >= 0))
        reinterpret_cast<uint16_t*>(routed ? g.out : g.out_shared)[(size_t)(routed ? my_pos : pair - S) * g.N + n] = (uint16_t)bits;
    auto row_value = [&](int q) { return __uint_as_float((uint32_t)__shfl((int)bits, (8 * q + f) & 63) << 16); };
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < M; ++q) {
        const float v = row_value(slot[q]);
        if (key[q] != 0x7fffffff) sum = __fadd_rn(sum, __fmul_rn(gate[q], v));
    }
    if (g.a_shared) sum = __fadd_rn(sum, row_value(S + token));
    if (g.cmb_residual) sum = __fadd_rn(sum, residual);
    if (tid < 8 * T) {
        if (g.cmb_f32) static_cast<float*>(g.cmb_out)[(size_t)token * g.N + n] = sum;
        else static_cast<bf16_t*>(g.cmb_out)[(size_t)token * g.N + n] = from_f32<bf16_t>(sum);
    }
}

// red_raw: TEAMS * NW * (SWIGLU ? 2 : 1) * 16 * kRedPitch floats of LDS; BATCH: reduction steps whose loads a wave issues together.
// TEAMS > 1: the workgroup is TEAMS teams of NW waves, each with a feature block `fb` of its own (the caller hands
// every team its block; a team without one has left the kernel before: the barrier below counts the waves that
// are still there).
// LATE_ROWS: which rows the side has is looked at behind the first weight loads (`late`); a side without rows leaves
// with sd.rows == 0 and nothing stored, and row r is stored at its slot.
// hook(): what the workgroup does between the first weight loads and the first look at a row (every wave runs it once; it
// leaves everything it puts into LDS behind a barrier, and `red_raw` free).
template <bool SWIGLU, bool I8, int NW, int BATCH, int TEAMS, bool LATE_ROWS, typename ROWS, typename HOOK>
__device__ __forceinline__ void decode_gemm_body(DecodeSide& sd, int fb, float* red_raw, LateRows* late, HOOK hook) {
    const int team = TEAMS > 1 ? (int)threadIdx.x / (NW * 64) : 0;
    float (*red)[SWIGLU ? 2 : 1][16][kRedPitch] =
        reinterpret_cast<float (*)[SWIGLU ? 2 : 1][16][kRedPitch]>(red_raw + (size_t)team * NW * (SWIGLU ? 2 : 1) * 16 * kRedPitch);
    const int tid = (int)threadIdx.x - team * (NW * 64);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = sd.K;
    const int steps = K / 16;
    const int chunk = (steps + NW - 1) / NW;
    const int g0 = min(steps, wave * chunk), g1 = min(steps, g0 + chunk);

    // packed weights: row block rb starts at rb * K * 32 elements; step s, lane l at (s * 64 + l) * 16 bytes
    // (int8: steps come in pairs, 16 bytes per lane and pair, the even step first)
    const size_t block_bytes = (size_t)K * 32 * (I8 ? 1 : 2);
    const char* w0 = sd.w + (size_t)fb * block_bytes;
    const char* w1 = sd.w + (size_t)(sd.N / 32 + fb) * block_bytes;  // the matching up rows
    auto wfrag = [&](const char* base, int s) -> bf16x8 {
        if constexpr (I8) {
            const uint2 q = *reinterpret_cast<const uint2*>(base + ((size_t)(s >> 1) * 64 + lane) * 16 + (s & 1) * 8);
            return widen_i8(q);
        } else {
            const uint4 q = *reinterpret_cast<const uint4*>(base + ((size_t)s * 64 + lane) * 16);
            return __builtin_bit_cast(bf16x8, q);
        }
    };
    // token fragment: lane -> token lane % 32, columns 16 s + 8 (lane / 32) .. + 7
    int grow = 0;
    if constexpr (!LATE_ROWS) {
        const int trow = (lane & 31) < sd.rows ? (lane & 31) : 0;
        grow = (sd.row_index ? sd.row_index[sd.row0 + trow] : sd.row0 + trow) + sd.a_row0;  // awaited after the weight loads
    }

    // int8: the scales of the four features this thread will finish, under way before the weights
    float4 sc0 = make_float4(1.0f, 1.0f, 1.0f, 1.0f), sc1 = sc0;
    if constexpr (I8) {
        sc0 = *reinterpret_cast<const float4*>(sd.scales + fb * 32 + 4 * (tid & 7));
        if constexpr (SWIGLU) sc1 = *reinterpret_cast<const float4*>(sd.scales + sd.N + fb * 32 + 4 * (tid & 7));
    }

    floatx16 acc0, acc1;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc0[v] = acc1[v] = 0.0f;
    float row_factor = 1.0f;  // ROWS::kNorm: of this lane's token
    int slot_expert[LATE_ROWS ? kLateRounds : 1];  // lane l: the experts of slots l, l + 64, ... (past the last: nobody's)
    if constexpr (LATE_ROWS) {
#pragma unroll
        for (int i = 0; i < kLateRounds; ++i) slot_expert[i] = late->expert_of[min(lane + 64 * i, late->S - 1)];
    }

    // One batch of reduction steps.  The first batch stands in front of the loop over the others, as straight
    // code: at the head of a loop the compiler waits for every load still under way - the row index, what the
    // combine fetched early - before the first weight load could go out.  Returns true when the side has no rows.
    auto batch = [&](const int s0, auto first_tag) -> bool {
        constexpr bool kFirst = decltype(first_tag)::value;
        bf16x8 wa[BATCH], wb[BATCH];
        uint4 raw[BATCH][ROWS::kPlain || sizeof(typename ROWS::type) == 2 ? 1 : 2];
        // the weights first: the address of a token row depends on a load of its own (the row index), and
        // loads are issued in order - nothing of the stream may queue up behind that wait
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const int s = min(s0 + u, g1 - 1);
            wa[u] = wfrag(w0, s);
            if constexpr (SWIGLU) wb[u] = wfrag(w1, s);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (LATE_ROWS && kFirst) {
            if (late->routed) {
                // the expert's rows in slot order: a matching lane pushes its slot to the lane numbered by the row
                int rows = 0, slot = 0;
#pragma unroll
                for (int i = 0; i < kLateRounds; ++i) {
                    if (64 * i >= late->S) break;  // uniform
                    const bool mine = lane + 64 * i < late->S && slot_expert[i] == late->expert;
                    const unsigned long long m = __ballot(mine);
                    const int rank = rows + __popcll(m & ((1ull << lane) - 1ull));  // below 32: a token names an expert once
                    const int pushed = __builtin_amdgcn_ds_permute(4 * (mine ? rank : 63), lane + 64 * i);
                    const int upto = rows + __popcll(m);
                    slot = lane >= rows && lane < upto ? pushed : slot;
                    rows = upto;
                }
                sd.rows = rows;
                if (rows <= 0) return true;  // the whole workgroup
                if (wave == 0 && lane < 32) late->row_slot[lane] = slot;
                const int trow = (lane & 31) < rows ? (lane & 31) : 0;
                const int mine_slot = __shfl(slot, trow);
                grow = mine_slot / late->k + sd.a_row0;
            } else {
                if (sd.rows <= 0) return true;
                grow = sd.row0 + ((lane & 31) < sd.rows ? (lane & 31) : 0);
            }
        }
        // (the empty statement pins the first use of the row index, and with it the wait for it, below the
        // weight loads; the barriers keep every load of the batch ahead of the first multiply)
        asm volatile("" : "+v"(grow));
        const typename ROWS::type* arow = reinterpret_cast<const typename ROWS::type*>(sd.a) + (size_t)grow * K + 8 * (lane >> 5);
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const int s = min(s0 + u, g1 - 1);
            const uint4* const from = reinterpret_cast<const uint4*>(arow + 16 * s);
            raw[u][0] = from[0];
            if constexpr (sizeof(typename ROWS::type) == 4) raw[u][1] = from[1];
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kFirst && !std::is_same<HOOK, NoHook>::value) {
            if constexpr (I8) {
                if (sd.widen_first) {  // uniform over the wave: it has nothing else to do before the rows are normed
#pragma unroll
                    for (int u = 0; u < BATCH; ++u) {
                        asm volatile("" : "+v"(wa[u]));
                        if constexpr (SWIGLU) asm volatile("" : "+v"(wb[u]));
                    }
                }
            }
            hook();
            if constexpr (ROWS::kNorm) row_factor = sd.row_factor[lane & 31];
        }
        auto fragment = [&](int u) -> bf16x8 {
            if constexpr (ROWS::kPlain) {
                return __builtin_bit_cast(bf16x8, raw[u][0]);
            } else {
                float v[8];
                if constexpr (sizeof(typename ROWS::type) == 2) {
                    Vec16<bf16_t>::widen(raw[u][0], v);
                } else {
                    float lo[4], hi[4];
                    Vec16<float>::widen(raw[u][0], lo);
                    Vec16<float>::widen(raw[u][1], hi);
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = lo[q], v[4 + q] = hi[q];
                }
                if constexpr (ROWS::kNorm) {
                    const float* const nw = sd.norm_w + 16 * (s0 + u) + 8 * (lane >> 5);
                    const float4 na = *reinterpret_cast<const float4*>(nw), nb = *reinterpret_cast<const float4*>(nw + 4);
                    const float n[8] = {na.x, na.y, na.z, na.w, nb.x, nb.y, nb.z, nb.w};
#pragma unroll
                    for (int q = 0; q < 8; ++q) v[q] = __fmul_rn(__fmul_rn(v[q], row_factor), n[q]);
                }
                return __builtin_bit_cast(bf16x8, make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])));
            }
        };
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            if (s0 + u < g1) {
                const bf16x8 tf = fragment(u);
                acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa[u], tf, acc0, 0, 0, 0);
                if constexpr (SWIGLU) acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wb[u], tf, acc1, 0, 0, 0);
            }
        }
        return false;
    };
    // (LATE_ROWS: every wave takes the first batch, also one without a reduction step of its own, so that all of
    // them learn the rows and leave together when there are none)
    if (LATE_ROWS || ROWS::kNorm || g0 < g1) {
        if (batch(g0, std::true_type{})) return;
    }
    for (int s0 = g0 + BATCH; s0 < g1; s0 += BATCH) batch(s0, std::false_type{});
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        red[wave][0][v][lane] = acc0[v];
        if constexpr (SWIGLU) red[wave][1][v][lane] = acc1[v];
    }
    __syncthreads();
    // accumulator element v of lane l: feature 8 (v / 4) + 4 (l / 32) + v % 4, token l % 32;
    // the partial sums of the waves are added in wave order.  A thread takes four neighbouring features of one token
    // and eight neighbouring threads one token's 32 features of the block: a row segment of 64 bytes leaves as one
    // piece (rows that another workgroup of the launch reads go through to memory, where a write of a few bytes
    // costs what a whole segment does).
    if (tid < 256) {
        const int token = tid >> 3, q = tid & 7;
        const int v = 4 * (q >> 1), l = token + 32 * (q & 1), f = 4 * q;
        if (token < sd.rows) {
            float y4[4];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                float y = red[0][0][v + h][l];
#pragma unroll
                for (int w = 1; w < NW; ++w) y += red[w][0][v + h][l];
                if constexpr (I8) y *= h == 0 ? sc0.x : h == 1 ? sc0.y : h == 2 ? sc0.z : sc0.w;
                if constexpr (SWIGLU) {
                    float u = red[0][1][v + h][l];
#pragma unroll
                    for (int w = 1; w < NW; ++w) u += red[w][1][v + h][l];
                    if constexpr (I8) u *= h == 0 ? sc1.x : h == 1 ? sc1.y : h == 2 ? sc1.z : sc1.w;
                    y = silu_bf16_grade(y) * u;
                }
                y4[h] = y;
            }
            int out_row = sd.out_row0 + sd.row0 + token;
            if constexpr (LATE_ROWS)
                if (late->routed) out_row = late->row_slot[token];
            bf16_t* const where = sd.out + (size_t)out_row * sd.N + fb * 32 + f;
            const unsigned long long four =
                (unsigned long long)((uint32_t)f32_to_bf16_bits(y4[0]) | ((uint32_t)f32_to_bf16_bits(y4[1]) << 16)) |
                ((unsigned long long)((uint32_t)f32_to_bf16_bits(y4[2]) | ((uint32_t)f32_to_bf16_bits(y4[3]) << 16)) << 32);
            if (sd.coherent_out)
                __hip_atomic_store(reinterpret_cast<unsigned long long*>(where), four, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else
                *reinterpret_cast<unsigned long long*>(where) = four;
        }
    }
}

// ---------------------------------------------------------------------------
// decode_front_kernel: norm, routing and the gate/up products in ONE launch, side by side.
// The gate/up product of a routed expert needs nothing of the routing but WHICH rows the expert takes.  With at most 32
// tokens an expert's rows are one tile whatever the routing says, so every expert's gate/up product is taken over ALL
// the call's rows - hidden rows [E][T, F] - without waiting for the routing: an expert that turns out unrouted costs its
// weights' bytes (the caller weighs them against the launch and the chain that this saves), the rows nobody routed to an
// expert cost nothing (the tile is 32 rows either way).  The first workgroups route, eight tokens each (route_rows_body);
// the others take two feature blocks of one side each: experts 0 .. E-1, then the shared expert's 32-row blocks.  The
// products read the call's own rows: a norm in front of the layer is applied on the way (RowForm), f32 rows are rounded.
// The down product then picks the routed rows out of the per-expert hidden rows (DecodeGemmArgs::a_expert_rows).
// ---------------------------------------------------------------------------
// A routing workgroup's tokens.  (1, 2 or 4: the same times with 8 rows by bf16 weights, where the products take longer than the
// routing.  Over int8 weights behind a norm the routing is the longer part, 12.8 us of a launch whose products end before; not timed.)
constexpr int kFrontTokens = 8;
constexpr int kFrontTeams = 2;   // feature blocks of a product workgroup
constexpr int kFrontRedFloats = kFrontTeams * 4 * 2 * 16 * kRedPitch;  // a product workgroup's partial sums
// ... which share their room with the rows' squares of a call behind a norm (d + 4 floats a row; 64: the chain reads ahead)
__host__ __device__ static int front_room_floats(int T, int d, bool norm) {
    const int squares = norm && !(T <= 8 && wave_norms(d)) ? T * (d + 4) + 64 : 0;
    return squares > kFrontRedFloats ? squares : kFrontRedFloats;
}

template <typename XT, bool I8, bool Q8, bool NORM>
__global__ __launch_bounds__(kSmallThreads, 2) void decode_front_kernel(RouteRowsArgs r, DecodeGemmArgs g, int routers) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int E = r.E, T = r.T;
    if ((int)blockIdx.x < routers) {
        const int k = r.k, ES = E | 1;
        const int t0 = blockIdx.x * kFrontTokens, nt = min(kFrontTokens, T - t0);
        float* const prob = reinterpret_cast<float*>(lds);  // the arrays of router_fixed_bytes
        float* const lsev = prob + kFrontTokens * ES;
        int* const lexp = reinterpret_cast<int*>(lsev + kFrontTokens);
        const RouteOut out{r.P, r.lse, r.expert_of, r.gate_of};
        if constexpr (sizeof(XT) == 2)
            if (r.exact) {  // uniform over the launch
                ExactLogits<kFrontTokens, Q8 ? 32 : 8> logits(r, lds);
                logits.folded = !route_exact_body<kFrontTokens, Q8 ? 32 : 8, NORM>(r, blockIdx.x, 0, E, true, lds);
                if (logits.folded) __syncthreads();
                block_softmax_topk<1, kFrontTokens>(prob, lsev, lexp, t0, nt, r.valid, E, k, out, logits);
                return;
            }
        route_rows_body<XT, kFrontTokens, Q8 ? 32 : 8, Q8 ? 2 : 1, 2, NORM>(r, blockIdx.x, 0, E, lds);
        __syncthreads();
        block_softmax_topk<1, kFrontTokens>(prob, lsev, lexp, t0, nt, r.valid, E, k, out, [&](int i, int e) { return prob[i * ES + e]; });
        return;
    }
    // a product workgroup is two teams of four waves, each with a block of 32 features of its own: the reduction is
    // split four ways as in the launch without the routing, and a compute unit has twice the weight bytes in flight
    const int widest = g.a_shared ? max(g.N, g.N_shared) : g.N;
    const int nfb = widest / 32, npair = (nfb + kFrontTeams - 1) / kFrontTeams;
    const int idx = blockIdx.x - routers;
    const int side = idx / npair;
    const int fb0 = kFrontTeams * (idx % npair);
    int fb = fb0 + (int)threadIdx.x / (kSmallThreads / kFrontTeams);
    DecodeSide sd;
    sd.row_index = nullptr;
    sd.row0 = 0;
    sd.a_row0 = 0;
    if (side < E) {
        sd.a = static_cast<const bf16_t*>(g.a);
        sd.w = static_cast<const char*>(g.w) + (size_t)side * g.w_expert_stride * (I8 ? 1 : 2);
        sd.scales = I8 ? g.scales + (size_t)side * g.s_expert_stride : nullptr;
        sd.out = static_cast<bf16_t*>(g.out);
        sd.N = g.N;
        sd.K = g.K;
        sd.rows = T;
        sd.out_row0 = side * T;
    } else {
        const int st = side - E;
        sd.a = static_cast<const bf16_t*>(g.a_shared);
        sd.w = static_cast<const char*>(g.w_shared);
        sd.scales = I8 ? g.scales_shared : nullptr;
        sd.out = static_cast<bf16_t*>(g.out_shared);
        sd.N = g.N_shared;
        sd.K = g.K_shared;
        sd.row0 = st * 32;
        sd.rows = min(32, g.T_shared - sd.row0);
        sd.out_row0 = 0;
    }
    if (fb0 * 32 >= sd.N) return;  // (the sides' widths differ)
    float* const red = reinterpret_cast<float*>(lds);
    if constexpr (NORM) {
        // (a team without a block keeps the other company to the barriers: it takes the last block again and stores nothing)
        if (fb * 32 >= sd.N) {
            fb = sd.N / 32 - 1;
            sd.rows = 0;
        }
        // The rows' factors are taken here as the routing takes them (route_rows_body), by every product workgroup for
        // itself: the rows are requested in front of the weights, squared and summed in index order while those stream in.
        const int d = r.d, sp = d + 4, tid = threadIdx.x;
        float* const nw = red + front_room_floats(T, d, true);
        float* const inv = nw + d;
        constexpr int NT = kSmallThreads;
        const float w0 = r.norm_w[min(tid, d - 1)], w1 = r.norm_w[min(tid + NT, d - 1)];
        auto put_norm_weights = [&]() {
            if (tid < d) nw[tid] = w0;
            if (tid + NT < d) nw[tid + NT] = w1;
            for (int c = tid + 2 * NT; c < d; c += NT) nw[c] = r.norm_w[c];
        };
        sd.norm_w = nw;
        sd.row_factor = inv;
        auto products = [&](auto hook) {
            decode_gemm_body<true, I8, kSmallThreads / 64 / kFrontTeams, sizeof(XT) == 4 ? 8 : kBatch, kFrontTeams, false,
                             RowForm<XT, NORM>>(sd, fb, red, nullptr, hook);
        };
        if (T <= 8 && wave_norms(d)) {
            // a wave a row (one token, d 512: the launch 7.6 us, 9.8 with a chain a thread; with four rows a wave, 32 tokens
            // of d 768, it is slower than the chains, 18.9 us a call against 18.6, for eight waves' sums share four units)
            const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
            const XT* const rows = static_cast<const XT*>(r.x);
            constexpr int MOST = 32 / Vec16<XT>::N;  // pieces a lane at most; of a shorter row the last one again
            const int most = d / 32 / Vec16<XT>::N - 1;
            struct Ahead {
                u32x4_t p[MOST];
            };
            auto fetch = [&](int row) {
                const u32x4_t* const from = reinterpret_cast<const u32x4_t*>(rows + (size_t)min(row, T - 1) * d + (tid & 31) * (d / 32));
                Ahead a;
#pragma unroll
                for (int p = 0; p < MOST; ++p) a.p[p] = from[min(p, most)];
                return a;
            };
            const Ahead own = fetch(wave);
            __builtin_amdgcn_sched_barrier(0);
            products([&]() {
                put_norm_weights();
                if (tid >= T && tid < 32) inv[tid] = 0.0f;
                if (wave < T)
                    with_lane_elements(d, [&](auto l_tag) {
                        LaneRow<XT, decltype(l_tag)::value> lr;
#pragma unroll
                        for (int p = 0; p < lr.P; ++p) lr.raw[p] = __builtin_bit_cast(uint4, own.p[p]);
                        const float f = lr.inverse_rms(r.norm_eps);
                        if ((tid & 63) == 0) inv[wave] = f;
                    });
                __syncthreads();
            });
            return;
        }
        // Squares in column order in LDS, a thread of the first wave a row.  The chain of additions is what the products wait
        // for, so nothing stands in front of it: seven waves lay down their share of the squares before they ask for any
        // weights, which then come in beside the chain, and the first wave asks for its own before its share (32 tokens, d 768,
        // int8: the launch 12.5 us with what else is said at kRedPitch; 15.4 with every wave's weights in front).
        const int xpr = d / Vec16<XT>::N, nx = T * xpr;
        const uint4* const xsrc = reinterpret_cast<const uint4*>(r.x);
        const uint32_t recip = (uint32_t)(0x100000000ull / (uint32_t)xpr) + 1u;
        auto lay_squares = [&]() {
            auto fetch = [&](int i) -> uint4 { return xsrc[(uint32_t)min(i, nx - 1)]; };
            auto put = [&](int i, const uint4& v) {
                if (i >= nx) return;
                const int row = xpr == 1 ? i : (int)__umulhi((uint32_t)i, recip), c = (i - row * xpr) * Vec16<XT>::N;
                float f[Vec16<XT>::N];
                Vec16<XT>::widen(v, f);
                float4* const s4 = reinterpret_cast<float4*>(red + row * sp + c);
#pragma unroll
                for (int q = 0; q < Vec16<XT>::N / 4; ++q)
                    s4[q] = make_float4(__fmul_rn(f[4 * q], f[4 * q]), __fmul_rn(f[4 * q + 1], f[4 * q + 1]),
                                        __fmul_rn(f[4 * q + 2], f[4 * q + 2]), __fmul_rn(f[4 * q + 3], f[4 * q + 3]));
            };
            for (int i = tid; i < nx; i += 6 * NT) {
                const uint4 v0 = fetch(i), v1 = fetch(i + NT), v2 = fetch(i + 2 * NT), v3 = fetch(i + 3 * NT), v4 = fetch(i + 4 * NT),
                            v5 = fetch(i + 5 * NT);
                __builtin_amdgcn_sched_barrier(0);
                put(i, v0); put(i + NT, v1); put(i + 2 * NT, v2);
                put(i + 3 * NT, v3); put(i + 4 * NT, v4); put(i + 5 * NT, v5);
            }
            put_norm_weights();
            __syncthreads();
        };
        const bool first_wave = __builtin_amdgcn_readfirstlane(tid >> 6) == 0;
        if (!first_wave) lay_squares();
        sd.widen_first = !first_wave;
        products([&]() {
            if (first_wave) {
                lay_squares();
                if (tid < T) inv[tid] = inverse_rms_of(ordered_sum(red + tid * sp, d), d, r.norm_eps);
                else if (tid < 32) inv[tid] = 0.0f;
            }
            __syncthreads();
        });
    } else {
        if (fb * 32 >= sd.N) return;
        // (f32 rows take two registers a fragment's worth: a shorter batch keeps everything in registers)
        decode_gemm_body<true, I8, kSmallThreads / 64 / kFrontTeams, sizeof(XT) == 4 ? 8 : kBatch, kFrontTeams, false,
                         RowForm<XT, NORM>>(sd, fb, red);
    }
}

// LDS of the launch; *EG: experts whose router rows a routing workgroup holds together.  0: the call does not fit.
static size_t front_lds_bytes(const RouterArgs& a, bool bf16, int* EG) {
    const int T = a.T, E = a.E, k = a.k, d = a.d;
    const bool q8 = a.wq != nullptr, norm = a.norm_w != nullptr, exact = route_exact_ok(a, bf16);
    const size_t products = ((size_t)front_room_floats(T, d, norm) + (norm ? d + 32 : 0)) * 4;
    int eg = E;
    auto route = [&] {
        return exact ? route_exact_lds_bytes(E, k, d, kFrontTokens, q8 ? 32 : 8, eg)
                     : route_rows_lds_bytes(E, k, d, kFrontTokens, q8 ? 32 : 8, eg, norm);
    };
    while (eg > (exact ? 16 : 8) && route() > (size_t)kMaxRouterLds)
        eg = exact ? exact_fewer(eg, kFrontTokens, q8 ? 32 : 8) : (eg - 1) & ~1;
    if (route() > (size_t)kMaxRouterLds || products > (size_t)kMaxRouterLds) return 0;
    *EG = eg;
    return products > route() ? products : route();
}

bool decode_front_ok(const RouterArgs& a, bool bf16) {
    const int unit = a.wq ? 32 : 8;
    const size_t xsize = bf16 ? 2 : 4;
    int eg = 0;
    return a.T >= 1 && a.T <= kSmallRouteMaxTokens && a.E <= 64 && a.k <= kMaxTopK && a.T * a.E <= kSmallRouteMaxPairs &&
           a.d % unit == 0 && a.d % 32 == 0 && (size_t)a.d * xsize % 16 == 0 && reinterpret_cast<uintptr_t>(a.x) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(a.wq ? static_cast<const void*>(a.wq) : a.wr) % 16 == 0 &&
           front_lds_bytes(a, bf16, &eg) != 0;
}

hipError_t launch_decode_front(const RouterArgs& a, const DecodeGemmArgs& g, bool bf16, WeightKind wk, hipStream_t s) {
    if (!decode_front_ok(a, bf16) || !g.swiglu || wk == WeightKind::F32 || (a.wq && (!a.wscale || wk != WeightKind::I8)))
        return hipErrorInvalidValue;
    const int shared_tiles = g.a_shared ? (g.T_shared + 31) / 32 : 0;
    const int widest = g.a_shared ? (g.N > g.N_shared ? g.N : g.N_shared) : g.N;
    const int routers = (a.T + kFrontTokens - 1) / kFrontTokens;
    const int grid = routers + (a.E + shared_tiles) * ((widest / 32 + kFrontTeams - 1) / kFrontTeams);
    int EG = 0;
    const size_t lds = front_lds_bytes(a, bf16, &EG);
    RouteRowsArgs r{a.x, a.wr, a.wq, a.wscale, a.bias, a.valid, a.T, a.d, a.E, a.k, EG, a.P, a.lse, a.expert_of, a.gate_of,
                    nullptr, nullptr, nullptr, nullptr, a.norm_w, a.norm_eps, nullptr, route_exact_ok(a, bf16), 0, nullptr,
                    a.exact_now};
    auto go = [&](auto kernel) -> hipError_t {
        static std::atomic<unsigned long long> attr_set{0};  // one per kernel: the lambda's body is instantiated for each
        const hipError_t e = once_per_device(attr_set, [&] {
            return hipFuncSetAttribute(reinterpret_cast<const void*>(+kernel.value), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       kMaxRouterLds);
        });
        if (e != hipSuccess) return e;
        RB_LAUNCH(kernel.value, dim3(grid), dim3(kSmallThreads), lds, s, r, g, routers);
        return hipGetLastError();
    };
#define RB_FRONT(XT, I8, Q8, NORM) \
    go(std::integral_constant<void (*)(RouteRowsArgs, DecodeGemmArgs, int), &decode_front_kernel<XT, I8, Q8, NORM>>{})
#define RB_FRONT_W(XT, NORM)                                                   \
    (wk == WeightKind::BF16 ? RB_FRONT(XT, false, false, NORM)                 \
                            : a.wq ? RB_FRONT(XT, true, true, NORM) : RB_FRONT(XT, true, false, NORM))
    if (bf16) return a.norm_w ? RB_FRONT_W(bf16_t, true) : RB_FRONT_W(bf16_t, false);
    return a.norm_w ? RB_FRONT_W(float, true) : RB_FRONT_W(float, false);
#undef RB_FRONT_W
#undef RB_FRONT
}

hipError_t launch_decode_layout(const DecodeLayoutArgs& a, hipStream_t s) {
    if (!small_route_ok(a.T, a.E, a.k)) return hipErrorInvalidValue;
    RB_LAUNCH(decode_layout_kernel, dim3(1), dim3(kSmallThreads), 0, s, a);
    return hipGetLastError();
}

constexpr int kByExpertSlots = 8;  // slots a token: what a thread of the combine fetches beforehand, and 64 * kLateRounds / 32

bool decode_down_by_expert_ok(const DecodeGemmArgs& g, int E, int T, int k) {
    return !g.swiglu && g.cmb_out != nullptr && g.cmb_counter != nullptr && g.cmb_gate_of != nullptr && g.a_expert_rows == T &&
           T >= 1 && T <= 32 && k <= kByExpertSlots && g.cmb_T == T && g.cmb_k == k && (!g.a_shared || g.N_shared == g.N) &&
           g.N / 32 <= kDecodeCombineMaxBlocks && g.N % 32 == 0 && E >= 1;
}

hipError_t launch_decode_down_by_expert(const DecodeGemmArgs& g, const DecodeLayoutArgs& t, WeightKind wk, hipStream_t s) {
    static_assert(kByExpertSlots * kSmallRouteMaxTokens <= 64 * kLateRounds, "every slot is looked at");
    if (!decode_down_by_expert_ok(g, t.E, t.T, t.k) || !small_route_ok(t.T, t.E, t.k)) return hipErrorInvalidValue;
    const int shared_tiles = g.a_shared ? (g.T_shared + 31) / 32 : 0;
    const dim3 grid(g.N / 32, t.E + shared_tiles + 1);
    const bool few = t.k <= 4;
    if (wk == WeightKind::BF16) {
        if (few) RB_LAUNCH((decode_down_by_expert_kernel<false, 4>), grid, dim3(512), 0, s, g, t);
        else RB_LAUNCH((decode_down_by_expert_kernel<false, kByExpertSlots>), grid, dim3(512), 0, s, g, t);
    } else if (wk == WeightKind::I8) {
        if (few) RB_LAUNCH((decode_down_by_expert_kernel<true, 4>), grid, dim3(512), 0, s, g, t);
        else RB_LAUNCH((decode_down_by_expert_kernel<true, kByExpertSlots>), grid, dim3(512), 0, s, g, t);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Up to four pairs.  (Eight, in two multiplies a step, were slower: two rows of the default model 14.5 against 13.8 us, four rows by
// 8 experts of 1408 19.2 against 15.0.)  int8 weights behind route_small_kernel stay with the tile table, which requests the weights
// no later: d 1024, 16 experts of 1408, 3 and 4 rows 30.7 and 31.4 us here, 30.4 and 31.1 there.
bool decode_down_few_ok(const DecodeGemmArgs& g, WeightKind wk, int T, int k) {
    const int pairs = T * (k + (g.a_shared ? 1 : 0));
    if (wk == WeightKind::F32 || (wk == WeightKind::I8 && g.a_expert_rows == 0)) return false;
    return !g.swiglu && g.cmb_out != nullptr && g.cmb_gate_of != nullptr && (g.a_expert_rows == 0 || g.a_expert_rows == T) && T >= 1 &&
           g.cmb_T == T && g.cmb_k == k && (!g.a_shared || g.N_shared == g.N) && g.N % 32 == 0 && pairs <= kFewPairs;
}

hipError_t launch_decode_down_few(const DecodeGemmArgs& g, const DecodeLayoutArgs& t, WeightKind wk, hipStream_t s) {
    if (!decode_down_few_ok(g, wk, t.T, t.k) || !small_route_ok(t.T, t.E, t.k)) return hipErrorInvalidValue;
    const dim3 grid(g.N / 8 + (g.a_expert_rows ? 1 : 0));
    auto go = [&](auto i8_tag) {
        constexpr bool I8 = decltype(i8_tag)::value;
        const int K = g.a_shared ? std::max(g.K, g.K_shared) : g.K, steps = (K / 16 + 7) / 8;
        if (steps <= 3) RB_LAUNCH((decode_down_few_kernel<I8, 3>), grid, dim3(512), 0, s, g, t);
        else if (steps <= 6) RB_LAUNCH((decode_down_few_kernel<I8, 6>), grid, dim3(512), 0, s, g, t);
        else RB_LAUNCH((decode_down_few_kernel<I8, 11>), grid, dim3(512), 0, s, g, t);
    };
    if (wk == WeightKind::I8) go(std::true_type{});
    else go(std::false_type{});
    return hipGetLastError();
}

bool decode_shape_ok(int N, int K) { return K % 32 == 0 && K >= 32 && N % 32 == 0 && N >= 32; }

hipError_t launch_decode_gemm(const DecodeGemmArgs& g, WeightKind wk, hipStream_t s) {
    const int shared_tiles = g.a_shared ? (g.T_shared + 31) / 32 : 0;
    const int tiles = g.max_tiles + shared_tiles;
    if (tiles <= 0) return hipSuccess;
    const int widest = g.a_shared ? (g.N > g.N_shared ? g.N : g.N_shared) : g.N;
    if (g.cmb_out != nullptr) {  // the combine rides on a down-shaped launch whose two sides have the same width
        if (g.swiglu || !g.cmb_counter || !g.cmb_inv_pos || !g.cmb_gate_of || (g.a_shared && g.N_shared != g.N) ||
            g.N / 32 > kDecodeCombineMaxBlocks || g.N % 2 != 0)
            return hipErrorInvalidValue;
    }
    const dim3 grid(widest / 32, tiles);
    if (wk == WeightKind::BF16) {
        if (g.swiglu) RB_LAUNCH((decode_gemm_kernel<true, false, 4>), grid, dim3(256), 0, s, g);
        else RB_LAUNCH((decode_gemm_kernel<false, false, 8>), grid, dim3(512), 0, s, g);
    } else if (wk == WeightKind::I8) {
        if (g.swiglu) RB_LAUNCH((decode_gemm_kernel<true, true, 4>), grid, dim3(256), 0, s, g);
        else RB_LAUNCH((decode_gemm_kernel<false, true, 8>), grid, dim3(512), 0, s, g);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace rbmoe
