// Where the routed slots go: the counting sort's scan over the router blocks' histograms, for the dispatch launch, and for
// gate/up products that do without one (RoutedSlots).
#pragma once

#include "rbmoe_kernels.h"

namespace rbmoe {

// ---- the whole layout, by a workgroup of at least 256 threads (all of them call it) ------------------------------------
__host__ __device__ static size_t layout_lds_bytes(int E) {
    const int parts = 256 / E;
    return ((size_t)2 * parts * E + (size_t)parts * (E + 1) + 4 * (size_t)(E + 1)) * 4;
}
struct LayoutSums {  // in LDS
    const int* off;   // [E + 1] first position of each expert
    const int* base;  // [E]     slots of each expert in the router blocks before `blk`
};
// Counts, offsets and the slots before router block `blk`; with `tables` counts, offsets and tile table are written, with
// `losses` the two auxiliary losses.
__device__ __forceinline__ LayoutSums layout_scan(const LayoutArgs& l, int blk, bool tables, bool loss_blk,
                                                  unsigned char* lds_raw) {
    const int* __restrict__ const blockcnt = l.blockcnt;
    const float* __restrict__ const partial = l.partial;
    const int T = l.T, E = l.E, k = l.k, TB = l.TB, tile_m = l.tile_m;
    const float w_aux = l.w_aux, w_z = l.w_z;
    int* const counts = l.counts;
    int* const offsets = l.offsets;
    int* const tile_expert = l.tile_expert;
    int* const tile_row0 = l.tile_row0;
    int* const tile_rows = l.tile_rows;
    int* const ntiles = l.ntiles;
    float* const losses = l.losses;
    const int parts = 256 / E;  // E <= 256
    int* const part_all = reinterpret_cast<int*>(lds_raw);           // [parts][E]
    int* const part_before = part_all + parts * E;                   // [parts][E]
    float* const part_mass = reinterpret_cast<float*>(part_before + parts * E);  // [parts][E+1] (losses)
    int* const cnt = reinterpret_cast<int*>(part_mass + parts * (E + 1));        // [E+1]
    int* const base = cnt + (E + 1);                                 // [E+1]
    int* const off = base + (E + 1);                                 // [E+1]
    float* const mass = reinterpret_cast<float*>(off + (E + 1));     // [E+1]
    const int tid = threadIdx.x;
    const int nb = (T + TB - 1) / TB;
    const int len = (nb + parts - 1) / parts;
    const int p = tid / E;
    const int e = tid - p * E;
    const bool active = p < parts;
    if (active) {
        const int b0 = min(nb, p * len), b1 = min(nb, b0 + len);
        // Loads in batches of 16 that do not depend on one another: one round trip to L2 per
        // batch instead of one per block.
        int s_all = 0, s_before = 0;
        float m = 0.0f, zs = 0.0f;
        for (int b = b0; b < b1; b += 16) {
            int c[16];
            float v[16], z[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) c[u] = blockcnt[(size_t)min(b + u, b1 - 1) * E + e];
            if (loss_blk) {
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    v[u] = partial[(size_t)min(b + u, b1 - 1) * (E + 1) + e];
                    z[u] = partial[(size_t)min(b + u, b1 - 1) * (E + 1) + E];
                }
            }
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                s_all += b + u < b1 ? c[u] : 0;
                s_before += b + u < min(blk, b1) ? c[u] : 0;
            }
            if (loss_blk) {
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    if (b + u < b1) {
                        m += v[u];
                        zs += z[u];
                    }
                }
            }
        }
        part_all[p * E + e] = s_all;
        part_before[p * E + e] = s_before;
        if (loss_blk) {
            part_mass[p * (E + 1) + e] = m;
            if (e == 0) part_mass[p * (E + 1) + E] = zs;
        }
    }
    __syncthreads();
    if (tid < E) {
        int ca = 0, cb = 0;
        float m = 0.0f;
        for (int q = 0; q < parts; ++q) {
            ca += part_all[q * E + tid];
            cb += part_before[q * E + tid];
            if (loss_blk) m += part_mass[q * (E + 1) + tid];
        }
        cnt[tid] = ca;
        base[tid] = cb;
        mass[tid] = m;
    }
    // the sum of lse^2 over the parts: by the last thread of the workgroup, which exists for every expert count
    // (a thread numbered E does not when E is the workgroup size) and owns no expert column unless E is 256
    if (loss_blk && tid == 255) {
        float zs = 0.0f;
        for (int q = 0; q < parts; ++q) zs += part_mass[q * (E + 1) + E];
        mass[E] = zs;
    }
    __syncthreads();
    if (E <= 64) {  // exclusive prefix over the experts: one wave, log2(64) shuffle steps
        if (tid < 64) {
            const int c = tid < E ? cnt[tid] : 0;
            int incl = c;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int up = __shfl_up(incl, o);
                if (tid >= o) incl += up;
            }
            if (tid < E) off[tid] = incl - c;
            if (tid == E - 1) off[E] = incl;
        }
    } else if (tid == 0) {
        int run = 0;
        for (int q = 0; q < E; ++q) {
            off[q] = run;
            run += cnt[q];
        }
        off[E] = run;
    }
    __syncthreads();
    if (tables) {
        if (tid < E) {
            counts[tid] = cnt[tid];
            offsets[tid] = off[tid];
            // tiles of this expert start after the tiles of the experts before it
            int first = 0;
            for (int q = 0; q < tid; ++q) first += (cnt[q] + tile_m - 1) / tile_m;
            const int n = (cnt[tid] + tile_m - 1) / tile_m;
            for (int i = 0; i < n; ++i) {
                tile_expert[first + i] = tid;
                tile_row0[first + i] = off[tid] + i * tile_m;
                tile_rows[first + i] = min(tile_m, cnt[tid] - i * tile_m);
            }
            if (tid == E - 1) ntiles[0] = first + n;
        }
        if (tid == 0) offsets[E] = off[E];
    }
    if (loss_blk) {
        // every valid token routes exactly k slots, so the valid-token count is routed / k.  The experts' terms
        // (two divisions and a product each) side by side, then their sum in expert order by one thread.
        const int V = off[E] / k;
        const float tokens = (float)V;
        const float slots = (float)V * (float)k;
        float* const term = part_mass;  // [E]: the parts' sums are used up
        if (tid < E && V > 0) term[tid] = ((float)cnt[tid] / slots) * (mass[tid] / tokens);
        __syncthreads();
        if (tid == 0) {
            float aux = 0.0f, z = 0.0f;
            if (V > 0) {
                for (int q = 0; q < E; ++q) aux = aux + term[q];
                aux = aux * ((float)E * w_aux);
                z = w_z * mass[E] / tokens;
            }
            losses[0] = aux;
            losses[1] = z;
        }
    }
    return {off, base};
}

// ---- one tile of the gate/up product ------------------------------------------------------------------------------------
// A workgroup finds out by itself which rows its tile has: the histograms (requested in one batch) give the experts' counts
// and with them the tile table's entry, the expert's column of them says which router blocks the tile's rows come from, and
// those blocks' slots, read once, say which rows they are.  That is one trip to memory behind the histograms, as many as
// tile table and row index take, and no launch in front.  Experts: a power of two up to 64 (a thread's pieces of the
// histograms then belong to one expert).
constexpr int kSlotsMaxHistogram = 4096;  // router blocks x experts
constexpr int kSlotsMaxBlocks = 1024;
constexpr int kSlotsTileM = 128;          // rows of a tile at most
struct SlotsLds {
    int hist[kSlotsMaxHistogram];
    int before[kSlotsMaxBlocks];  // slots of the tile's expert in the router blocks before each
    int wave_sum[8][64];
};

// Sums over the lanes up to and with each lane (a whole wave): inside rows of 16 lanes, then across them, all of it in the
// instructions' lane-permuting operand (six trips through LDS take three times as long).
__device__ __forceinline__ int sum_up_to_lane(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

struct RoutedTile {
    int expert, row0, rows, first;  // first: the tile's first row among its expert's
};
// The histograms and the tile table's length; the rest (lane = expert: its slots, the slots and tiles up to and with it) is for
// routed_tile.  Called by all NTH threads of the workgroup; when it returns every wave has the sums, so that a workgroup that
// does not go on to routed_tile (a dense tile) may use the LDS for something else.
struct RoutedCounts {
    int count, rows, tiles, ntiles;
};
template <int NTH>
__device__ __forceinline__ RoutedCounts routed_counts(const RoutedSlots& r, SlotsLds& lds) {
    const LayoutArgs& l = r.layout;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, E = l.E;
    const int n = ((l.T + l.TB - 1) >> r.tb_shift) * E;
    int sum = 0;
    auto batch = [&](auto count_tag) {
        constexpr int C = decltype(count_tag)::value;
        int v[C];
#pragma unroll
        for (int u = 0; u < C; ++u) v[u] = l.blockcnt[min(tid + NTH * u, n - 1)];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            lds.hist[tid + NTH * u] = v[u];  // (past the end: not read)
            sum += tid + NTH * u < n ? v[u] : 0;
        }
    };
    if (n <= 1024) batch(std::integral_constant<int, 1024 / NTH>{});
    else batch(std::integral_constant<int, kSlotsMaxHistogram / NTH>{});
    for (int o = E; o < 64; o <<= 1) sum += __shfl_xor(sum, o);
    lds.wave_sum[wave][lane] = sum;
    __syncthreads();
    RoutedCounts c;
    c.count = 0;
#pragma unroll
    for (int w = 0; w < NTH / 64; ++w) c.count += lds.wave_sum[w][lane];
    __syncthreads();
    c.count = lane < E ? c.count : 0;
    c.rows = sum_up_to_lane(c.count);
    c.tiles = sum_up_to_lane((c.count + l.tile_m - 1) >> r.tile_shift);
    c.ntiles = __builtin_amdgcn_readlane(c.tiles, E - 1);
    return c;
}
// Tile number `tm` of the tile table: its rows' tokens into `token` (in LDS, apart from `lds`, their slots behind them); with
// `tables` their entries of the permutation are written as well.  Called by all NTH threads; `token` is there when it returns and `lds` is free.
template <int NTH>
__device__ __forceinline__ RoutedTile routed_tile(const RoutedSlots& r, const RoutedCounts& c, int tm, bool tables, SlotsLds& lds,
                                                  int* token) {
    const LayoutArgs& l = r.layout;
    const int tid = threadIdx.x, lane = tid & 63, E = l.E, k = l.k;
    const int nb = (l.T + l.TB - 1) >> r.tb_shift;
    const unsigned long long past = __ballot(lane < E && c.tiles > tm);
    const int e = __ffsll((long long)past) - 1;
    const int count = __builtin_amdgcn_readlane(c.count, e);
    const int own_tiles = (count + l.tile_m - 1) >> r.tile_shift;
    RoutedTile t;
    t.expert = e;
    t.first = (tm - (__builtin_amdgcn_readlane(c.tiles, e) - own_tiles)) * l.tile_m;
    t.row0 = __builtin_amdgcn_readlane(c.rows, e) - count + t.first;
    t.rows = min(l.tile_m, count - t.first);
    // the expert's column: a lane takes nbl blocks that follow one another (every wave for itself)
    const int nbl = (nb + 63) / 64, b0 = lane * nbl;
    int own = 0;
    for (int i = 0; i < nbl; ++i)
        if (b0 + i < nb) own += lds.hist[(b0 + i) * E + e];
    const int incl = sum_up_to_lane(own);
    int run = incl - own;
    const unsigned long long has = __ballot(own > 0 && run < t.first + t.rows && incl > t.first);  // blocks with rows of the tile
    for (int i = 0; i < nbl; ++i)
        if (b0 + i < nb) {
            lds.before[b0 + i] = run;
            run += lds.hist[(b0 + i) * E + e];
        }
    const int S = l.T * k;
    const int lane_slots = (nbl << r.tb_shift) * k;
    const int from = (__ffsll((long long)has) - 1) * lane_slots, to = min(S, (64 - __clzll((long long)has)) * lane_slots);
    __syncthreads();
    constexpr int U = 8;
    for (int s0 = from + tid; s0 < to; s0 += NTH * U) {
        int ex[U], rank[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = min(s0 + NTH * u, to - 1);
            ex[u] = r.expert_of[s];
            rank[u] = r.rank_in_block[s];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = s0 + NTH * u;
            if (s >= to || ex[u] != e) continue;
            const int tok = k == 1 ? s : (int)__umulhi((uint32_t)s, r.k_recip);
            const int pos = lds.before[tok >> r.tb_shift] + rank[u] - t.first;
            if (pos < 0 || pos >= t.rows) continue;
            token[pos] = tok;
            token[kSlotsTileM + pos] = s;
        }
    }
    __syncthreads();
    if (tables && tid < t.rows) {
        const int s = token[kSlotsTileM + tid];
        r.perm_slot[t.row0 + tid] = s;
        r.perm_token[t.row0 + tid] = token[tid];
        r.inv_pos[s] = t.row0 + tid;
    }
    return t;
}
// What no tile writes: the tables of the whole call, and the slots that go nowhere.  A workgroup of its own.
__device__ __forceinline__ void routed_rest(const RoutedSlots& r, unsigned char* lds_raw) {
    const int S = r.layout.T * r.layout.k;
    for (int s = threadIdx.x; s < S; s += blockDim.x)
        if (r.expert_of[s] < 0) r.inv_pos[s] = -1;
    layout_scan(r.layout, 0, true, true, lds_raw);
}

}  // namespace rbmoe
