// Grouped expert products for all-f32 layers on the f32 matrix cores of gfx950
// (v_mfma_f32_32x32x2_f32: f32 products, f32 accumulation).
//
//   out[row, n] = sum_c a[row, c] * w[expert][n, c]                 (down product)
//   out[row, n] = silu(a . wgate[n]) * (a . wup[n])                 (gate/up product)
//
// A workgroup owns 64 or 32 token rows x 64 output features; a wave owns 32 x 32 of them (gate/up: two
// accumulators, the gate rows and the matching up rows).  Both operands go global -> LDS by LDS-DMA in slices of SK
// reduction columns; one 16-byte LDS read per operand feeds four multiplies, the next fragments and the next slices
// are under way while a fragment is multiplied.  With SPLIT = 2 the workgroup has two groups of 4 waves that take
// the two halves of every slice and add their accumulators through LDS at the end (group 1 first, then group 0
// on top: a fixed order): twice the waves for the same tiles, which is what a launch with few tiles needs.
//
// Exactly two waves a SIMD (amdgpu_waves_per_eu): the kernel needs 86 registers at most, and where more waves may be
// resident the hardware fills some SIMDs with three or more while others hold one - a kernel of nothing but multiplies
// falls from 156 to 103 TFLOP/s that way (512 workgroups of 4 waves, one or two accumulators each).  One wave a SIMD
// leaves a workgroup's first loads and its stores uncovered.  What remains is the clock: the launch runs at 2.16 GHz
// (multiplies alone on random data: 130-141 TFLOP/s), and the last round of a launch.
// 1024 tokens, d 512, 8 experts top-2 of width 1408: gate/up 76.6 -> 73.7 us, down 51.6 -> 43.7 us (68 TFLOP/s); 8192
// tokens: 463 -> 451 and 256 -> 236 us (105 and 100 TFLOP/s).  Same box, against the kernel that staged through
// registers with one LDS stage, 4-byte fragment reads and three workgroups a compute unit.  One wave a SIMD: 76.8 / 48.8
// and 469 / 263 us; three: 77.1 / 47.8 and 470 / 244; 32 x 32 tiles with four wave groups 83.8 / 45.6.  A layer's output
// against 64 bits: 6.46e-7 (6.48e-7 before), 9.16e-7 (the same) at 8192 tokens.
// Rows are fetched through `row_index`, so the gather of
// the routed rows (gather_rows, src/moe.rs:658-664) never materialises.  The weight fragment
// is the matrix-core A operand and the token fragment B, so a lane ends with 4 consecutive
// features of one token (one 16-byte store).  SiLU uses the exact division: this path is held
// to 1e-5.  For a backward pass the gate/up launch can also keep the pre-activations (`gu_out`),
// and a plain launch can apply SwiGLU's backward where it stores its rows (`swiglu_grad_gu`).
#include <type_traits>

#include "rbmoe_kernels.h"

namespace rbmoe {

namespace {

constexpr int FN = 64;   // output features per workgroup (two waves side by side)
constexpr int FK = 32;   // reduction widths are multiples of this

// Loads go to LDS by LDS-DMA, issued from inline assembly: the compiler would drain every load in flight in front of
// an LDS read otherwise.  A wave deposits 64 pieces of 16 bytes at consecutive LDS addresses.
__device__ __forceinline__ void f32_issue_dma(uint32_t lds_addr, const float* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_addr), "v"(src) : "memory");
}
template <int N>
__device__ __forceinline__ void f32_wait_outstanding() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// FM = token rows per workgroup, 64 or 32 (FM / 32 x 2 waves per group); SPLIT = wave groups; SK = reduction columns of
// a slice, SK / SPLIT of them multiplied by each wave group; STAGES = LDS stages of one slice each
template <bool SWIGLU, int FM, int SPLIT, int SK, int STAGES>
__global__ __launch_bounds__(FM * 4 * SPLIT) __attribute__((amdgpu_waves_per_eu(2, 2))) void grouped_f32_kernel(
    const float* __restrict__ a, const int* __restrict__ row_index, const float* __restrict__ w,
    size_t w_expert_stride, int N, int K, const int* __restrict__ tile_expert, const int* __restrict__ tile_row0,
    const int* __restrict__ tile_rows, const int* __restrict__ ntiles, int dense_rows, float* __restrict__ out,
    float* __restrict__ gu_out, const float* __restrict__ bw_gu) {
    constexpr int WR = SWIGLU ? 2 * FN : FN;  // weight rows staged per slice
    constexpr int WPG = FM / 32 * 2;          // waves per group
    constexpr int NTH = 64 * WPG * SPLIT;     // threads
    constexpr int NW = NTH / 64;
    constexpr int PPR = SK / 4;               // 16-byte pieces per staged row: 4 or 8
    constexpr int STAGE = (FM + WR) * SK;     // floats of a stage: token rows, then weight rows
    constexpr int STEPS = SK / SPLIT / 8;     // fragment reads (four multiplies deep) per slice and wave
    constexpr int DMA = (FM + WR) * PPR / 64 / NW;  // LDS-DMA instructions per wave and slice
    static_assert(DMA * 64 * NW == (FM + WR) * PPR && STEPS % 2 == 0, "whole instructions, two fragment sets in turn");
    __shared__ __attribute__((aligned(16))) float lds[STAGES * STAGE];

    // ---- which tile: each XCD (workgroup number mod 8) walks a contiguous range of tiles with one expert's row tiles
    // innermost, so that a weight slice is fetched by one L2 (in grid order every slice was fetched by four or eight)
    const int tiles_n = (N + FN - 1) / FN;
    const int tiles_m = dense_rows >= 0 ? (dense_rows + FM - 1) / FM : *ntiles;
    const int total = tiles_m * tiles_n;
    const int per_xcd = (total + 7) / 8;
    const int local = blockIdx.x >> 3;
    if (local >= per_xcd) return;
    const int pid = (blockIdx.x & 7) * per_xcd + local;
    if (pid >= total) return;
    constexpr int GROUP_M = 8;
    const int per_group = GROUP_M * tiles_n;
    const int first_m = pid / per_group * GROUP_M;
    const int gsize = min(GROUP_M, tiles_m - first_m);
    const int in_g = pid % per_group;
    const int tm_idx = first_m + in_g % gsize;
    const int n0 = in_g / gsize * FN;

    int expert, row0, rows;
    if (dense_rows >= 0) {
        expert = 0;
        row0 = tm_idx * FM;
        rows = min(FM, dense_rows - row0);
    } else {
        expert = tile_expert[tm_idx];
        row0 = tile_row0[tm_idx];
        rows = tile_rows[tm_idx];
    }
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wv % WPG;
    const int grp = wv / WPG;                 // wave group: which part of each slice it multiplies
    const int wy = wave >> 1, wx = wave & 1;  // token half, feature half
    const float* wbase = w + (size_t)expert * w_expert_stride;

    // ---- staging: instruction i of a wave fills LDS pieces 64 (wv DMA + i) .. + 63 of the stage.  Rows cannot be
    // padded apart, so position q of row r holds piece q ^ swz(r): the 16 rows that 16 lanes of a fragment read touch
    // at one logical piece then lie in 64 distinct banks.
    auto swz = [](int r) { return PPR == 8 ? ((r >> 1) & 7) : ((r >> 2) & 3); };
    const float* src[DMA];
#pragma unroll
    for (int i = 0; i < DMA; ++i) {
        const int p = (wv * DMA + i) * 64 + lane;
        const int r = p / PPR;                    // row of the stage
        const int c = 4 * ((p % PPR) ^ swz(r));   // swz(FM + r) == swz(r): FM is a multiple of 16
        if (r < FM) {
            const int rr = r < rows ? r : 0;  // rows past the end of the group: products never stored
            const int grow = row_index ? row_index[row0 + rr] : row0 + rr;
            src[i] = a + (size_t)grow * K + c;
        } else {
            // weight row q < FN: gate (or plain) feature n0 + q; q >= FN: the matching up row
            const int q = r - FM;
            const int feat = n0 + (q % FN);
            const int fr = feat < N ? feat : 0;
            src[i] = wbase + (size_t)((SWIGLU && q >= FN) ? N + fr : fr) * K + c;
        }
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)wv * (DMA * 1024);
    const int KT = K / SK;
    auto dma = [&](int kt, int stage) {
        const int k0 = min(kt, KT - 1) * SK;  // past the end: fetched again and never read, so that the wait counts hold
#pragma unroll
        for (int i = 0; i < DMA; ++i) f32_issue_dma(lds0 + (uint32_t)(stage * (STAGE * 4) + i * 1024), src[i] + k0);
    };

    floatx16 acc0, acc1;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc0[v] = acc1[v] = 0.0f;

    // ---- fragments: one 16-byte read per operand feeds four multiplies.  Lane l reads row l % 32 of the wave's block,
    // the columns 8 s + 4 (l / 32) .. + 3 of the group's share of the slice; multiply j takes column j of both halves
    // (both operands in the same order, so the product is the same sum).
    const int frow = lane & 31, fhalf = lane >> 5;
    const int fsw = swz(frow);
    const float* const a_rows = lds + (wy * 32 + frow) * SK;
    const float* const w_rows = lds + (FM + wx * 32 + frow) * SK;
    struct Frag {
        float4 t, g, u;
    } fr[2];
    auto read = [&](Frag& f, int stage, int s) {
        const int o = stage * STAGE + 4 * ((grp * (PPR / SPLIT) + 2 * s + fhalf) ^ fsw);
        f.t = *reinterpret_cast<const float4*>(a_rows + o);
        f.g = *reinterpret_cast<const float4*>(w_rows + o);
        if constexpr (SWIGLU) f.u = *reinterpret_cast<const float4*>(w_rows + FN * SK + o);
    };
    auto mul = [&](float g, float u, float t) {
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(g, t, acc0, 0, 0, 0);
        if constexpr (SWIGLU) acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(u, t, acc1, 0, 0, 0);
    };

    // ---- main loop.  The one barrier of a slice stands in front of its last step, whose fragments are in registers by
    // then: before it a wave waits for its own DMA of the next slice (loads retire in order; STAGES - 2 younger slices
    // may be in flight), behind it the next slice is complete, its first fragments are read during this slice's last
    // multiplies, and this slice's stage, which nobody reads any more, takes the DMA of slice kt + STAGES.
    for (int i = 0; i < STAGES; ++i) dma(i, i);
    f32_wait_outstanding<(STAGES - 1) * DMA>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(fr[0], 0, 0);
    int st = 0;
    for (int kt = 0; kt < KT; ++kt) {
        const int nx = st + 1 == STAGES ? 0 : st + 1;
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            Frag& cur = fr[s & 1];
            if (s == STEPS - 1) {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"((STAGES - 2) * DMA) : "memory");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                read(fr[0], nx, 0);
                dma(kt + STAGES, st);
            } else {
                read(fr[(s + 1) & 1], st, s + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            mul(cur.g.x, SWIGLU ? cur.u.x : 0.0f, cur.t.x);
            mul(cur.g.y, SWIGLU ? cur.u.y : 0.0f, cur.t.y);
            mul(cur.g.z, SWIGLU ? cur.u.z : 0.0f, cur.t.z);
            mul(cur.g.w, SWIGLU ? cur.u.w : 0.0f, cur.t.w);
            __builtin_amdgcn_sched_barrier(0);
        }
        st = nx;
    }
    f32_wait_outstanding<0>();  // the LDS is used again below, and nothing may land after the workgroup has ended
    __syncthreads();

    if constexpr (SPLIT > 1) {
        // the two groups' sums meet in LDS (the staging tiles are free: the loop's last barrier is behind us)
        static_assert(STAGES * STAGE >= (SWIGLU ? 2 : 1) * WPG * 16 * 64, "room for the accumulators");
        float* const r0 = lds + wave * (16 * 64) + lane;
        float* const r1 = r0 + WPG * 16 * 64;
        // groups SPLIT - 1 ... 1 hand their sums down one after the other; group 0 adds the last and stores
#pragma unroll
        for (int gsrc = SPLIT - 1; gsrc >= 1; --gsrc) {
            if (grp == gsrc) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    r0[v * 64] = acc0[v];
                    if constexpr (SWIGLU) r1[v * 64] = acc1[v];
                }
            }
            __syncthreads();
            if (grp == gsrc - 1) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    acc0[v] += r0[v * 64];
                    if constexpr (SWIGLU) acc1[v] += r1[v * 64];
                }
            }
            if (gsrc > 1) __syncthreads();
        }
        if (grp != 0) return;
    }

    // accumulator element v of lane l: feature 8 (v / 4) + 4 (l / 32) + v % 4 of the wave's
    // block, token l % 32
    const int tok = wy * 32 + (lane & 31);
    if (tok >= rows) return;
    float* orow = out + (size_t)(row0 + tok) * N + n0 + wx * 32;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int f = 8 * q + 4 * (lane >> 5);
        if (n0 + wx * 32 + f >= N) continue;  // N is a multiple of 4: a group of 4 is in or out as a whole
        float4 y;
        if constexpr (SWIGLU) {
            y.x = silu_f32(acc0[4 * q + 0]) * acc1[4 * q + 0];
            y.y = silu_f32(acc0[4 * q + 1]) * acc1[4 * q + 1];
            y.z = silu_f32(acc0[4 * q + 2]) * acc1[4 * q + 2];
            y.w = silu_f32(acc0[4 * q + 3]) * acc1[4 * q + 3];
            if (gu_out != nullptr) {  // uniform: the pre-activations G | U [rows, 2 N] kept for a backward pass
                float* const grow = gu_out + (size_t)(row0 + tok) * 2 * N + n0 + wx * 32 + f;
                *reinterpret_cast<float4*>(grow) =
                    make_float4(acc0[4 * q + 0], acc0[4 * q + 1], acc0[4 * q + 2], acc0[4 * q + 3]);
                *reinterpret_cast<float4*>(grow + N) =
                    make_float4(acc1[4 * q + 0], acc1[4 * q + 1], acc1[4 * q + 2], acc1[4 * q + 3]);
            }
        } else {
            y = make_float4(acc0[4 * q + 0], acc0[4 * q + 1], acc0[4 * q + 2], acc0[4 * q + 3]);
            if (bw_gu != nullptr) {  // uniform
                // SwiGlu::backward (src/ffn.rs:87-120) on the way out: the product row is the gradient of the
                // hidden row; dG = dH * U * silu'(G), dU = dH * silu(G) go to `gu_out`, `out` is not written.
                const size_t off = (size_t)(row0 + tok) * 2 * N + n0 + wx * 32 + f;
                const float4 g4 = *reinterpret_cast<const float4*>(bw_gu + off);
                const float4 u4 = *reinterpret_cast<const float4*>(bw_gu + off + N);
                const float dh[4] = {y.x, y.y, y.z, y.w}, gv[4] = {g4.x, g4.y, g4.z, g4.w}, uv[4] = {u4.x, u4.y, u4.z, u4.w};
                float dg[4], du[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float sg = 1.0f / (1.0f + __expf(-gv[i]));
                    dg[i] = dh[i] * uv[i] * (sg * (1.0f + gv[i] * (1.0f - sg)));  // silu', src/ffn.rs:235-238
                    du[i] = dh[i] * (gv[i] * sg);
                }
                *reinterpret_cast<float4*>(gu_out + off) = make_float4(dg[0], dg[1], dg[2], dg[3]);
                *reinterpret_cast<float4*>(gu_out + off + N) = make_float4(du[0], du[1], du[2], du[3]);
                continue;
            }
        }
        *reinterpret_cast<float4*>(orow + f) = y;
    }
}

}  // namespace

// 64-row tiles; 32-row tiles when the launches of such a batch would have few tiles for the chip (their workgroups
// cannot be spread evenly over 256 compute units: 320 tiles leave a quarter of them with twice the work)
int f32_tile_m(int rows, int groups, int n_min) {
    const long long tiles64 = (long long)(rows / 64 + groups) * ((n_min + 63) / 64);
    return tiles64 < 4 * 256 ? 32 : 64;
}

// reduction width a multiple of the slice, output width a multiple of 4 (16-byte stores)
bool f32_shape_ok(int N, int K) { return K % FK == 0 && K >= FK && N % 4 == 0 && N >= 4; }

hipError_t launch_grouped_f32(const GroupedArgs& g, hipStream_t s) {
    // the tile table's tile height (a dense launch makes its own tiles: 64 rows, or 32 when that leaves few)
    int fm = g.tile_m;
    if (g.dense_rows >= 0) fm = f32_tile_m(g.dense_rows, 0, g.N);
    if (fm != 32 && fm != 64) return hipErrorInvalidValue;
    const int tiles_m = g.dense_rows >= 0 ? (g.dense_rows + fm - 1) / fm : g.max_tiles;
    if (tiles_m <= 0) return hipSuccess;
    const int total = (g.N + FN - 1) / FN * tiles_m;
    const dim3 grid((total + 7) / 8 * 8);
    auto go = [&](auto swiglu_tag, auto fm_tag, auto split_tag, auto sk_tag, auto stages_tag) {
        constexpr bool SW = decltype(swiglu_tag)::value;
        constexpr int FMv = decltype(fm_tag)::value, SP = decltype(split_tag)::value, SKv = decltype(sk_tag)::value,
                      ST = decltype(stages_tag)::value;
        RB_LAUNCH((grouped_f32_kernel<SW, FMv, SP, SKv, ST>), grid, dim3(FMv * 4 * SP), 0, s, static_cast<const float*>(g.a),
                  g.row_index, static_cast<const float*>(g.w), g.w_expert_stride, g.N, g.K, g.tile_expert, g.tile_row0,
                  g.tile_rows, g.ntiles, g.dense_rows, static_cast<float*>(g.out), static_cast<float*>(g.gu_out),
                  static_cast<const float*>(g.swiglu_grad_gu));
    };
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, 2> Two;
    typedef std::integral_constant<int, 3> Three;
    typedef std::integral_constant<int, 16> K16;
    typedef std::integral_constant<int, 32> K32;  // (and 32-row tiles)
    typedef std::integral_constant<int, 64> M64;
    // 32-row tiles have two waves per group: a second group brings the workgroup back to four
    if (fm == 64) {
        if (g.swiglu) go(std::true_type{}, M64{}, One{}, K16{}, Three{});
        else go(std::false_type{}, M64{}, One{}, K16{}, Three{});
    } else {
        if (g.swiglu) go(std::true_type{}, K32{}, Two{}, K32{}, Two{});
        else go(std::false_type{}, K32{}, Two{}, K32{}, Three{});
    }
    return hipGetLastError();
}

}  // namespace rbmoe
