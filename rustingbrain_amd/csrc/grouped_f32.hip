// Grouped expert products over f32 rows on the bf16 matrix cores of gfx950, at f32 accuracy.
//
//   out[row, n] = sum_c a[row, c] * w[expert][n, c]                 (down product)
//   out[row, n] = silu(a . wgate[n]) * (a . wup[n])                 (gate/up product)
//
// An f32 value of 2^-110 or more is the exact sum of three bf16 values, x = x1 + x2 + x3, each the nearest to what the ones
// before leave (24 bits of mantissa in three times eight, signs included).  Products of bf16 values are exact in f32, so
//   f32 weights    x w = x1 w1 + x1 w2 + x2 w1 + x1 w3 + x2 w2 + x3 w1 + (less than 2^-25 of |x w|): six multiplies on a
//                  unit of sixteen times the rate of the f32 one
//   bf16 weights   x w = x1 w + x2 w + x3 w, exactly: three
//   int8 weights   the same, the values being exact in bf16; the row's scale multiplies the sum (src/quantized.rs:55-62)
// with f32 accumulation.  A sum's error is that of its additions, and there are fewer of them than the f32 unit has (one
// a step of 16 columns for the large terms, the small ones summed apart or with them where the groups share out the
// steps): hidden rows against 64 bits, d 512, 8 experts of 1408, 1024 tokens, 1.9e-7 where v_mfma_f32_32x32x2 gave 4.3e-7,
// products over given rows 2.4e-7 / 4.8e-7; bf16 weights, width 352, 3.6e-7 where a chain of fused adds gave 6.2e-7.
// Rows and weights stay f32 in memory.
// bf16's smallest value is 2^-133: of a smaller f32 value than 2^-110 up to 2^-134 is lost, of the largest ones the first part
// rounds to infinity, and a product of first parts may be past the largest f32 where that of the values is not.  Sums that
// this could show in are taken again on the f32 unit (see `odd`): what is lost stays below 2^-44 of the row's largest value
// a product.  f32 weights below 2^-110 lose as much wherever their sum is 2^-90 or more, or zero.
//
// What bounds it.  A step of a 64 x 64 wave tile is 24 multiplies (768 cycles of the matrix core) and the splitting of two
// weight fragments (88 vector instructions, 352 cycles).  The rows are split once per workgroup, on their way from registers
// into three bf16 planes in LDS; weights go to LDS by LDS-DMA as they are and a wave splits its own fragments (nobody else
// needs them), so they take 4 bytes a value on every path.  Everything of a step sits between its multiplies, one piece
// behind each (see `step`).  Large launches run at the power limit: 8192 tokens, same layer, gate/up 451 -> 288 us (the
// six bf16 products at 985 TFLOP/s, where the library's large bf16 product reaches 1160), down 236 -> 163; 1024 tokens
// 75 -> 47 and 44 -> 31, against the kernel on the f32 unit (of the large launches 1 % is the look at the rows' largest values
// and the sums' sizes, of the smallest 0.2 us).  Small ones are a chain of slices and memory: see f32_tile.
// f32 rows over bf16 or int8 weights at widths off 64 ran on the any-shape kernel's 20 TFLOP/s: 52 rows, d 768, 32 experts
// of 352 and a shared one 154 -> 58 us a forward.
//
// Rows are fetched through `row_index`, so the gather of the routed rows (gather_rows, src/moe.rs:658-664) never
// materialises.  The weight fragment is the matrix-core A operand and the token fragment B, so a lane ends with 4
// consecutive features of one token.  SiLU uses the exact division: this path is held to 1e-5.  For a backward pass the
// gate/up launch can also keep the pre-activations (`gu_out`), and a plain launch can apply SwiGLU's backward where it
// stores its rows (`bw_gu`).
#include <algorithm>
#include <type_traits>

#include "layout_device.h"
#include "rbmoe_kernels.h"

namespace rbmoe {

namespace {

constexpr int RING = 3;   // LDS stages of weights

// Every load of the main loop is issued from inline assembly and awaited by a hand-counted vmcnt: the compiler would drain
// all loads in flight in front of an LDS read otherwise.  An LDS-DMA deposits 64 pieces of 16 bytes at consecutive
// addresses.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void f32_issue_dma(uint32_t lds_addr, const void* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_addr), "v"(src) : "memory");
}
__device__ __forceinline__ void f32_issue_load(u32x4& d, const void* src) {
    asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(d) : "v"(src));
}

template <int I, int N, typename F>
__device__ __forceinline__ void f32_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        f32_for<I + 1, N>(f);
    }
}

// Two f32 values as three pairs of bf16: nearest, nearest of the rest, the rest.
__device__ __forceinline__ void split2(float x, float y, uint32_t& a, uint32_t& b, uint32_t& c) {
    a = pack2(x, y);
    const float x1 = x - __uint_as_float(a << 16), y1 = y - __uint_as_float(a & 0xffff0000u);
    b = pack2(x1, y1);
    c = pack2(x1 - __uint_as_float(b << 16), y1 - __uint_as_float(b & 0xffff0000u));
}

// Magnitudes in the order of their values, a NaN above all of them.
__device__ __forceinline__ uint32_t magnitude(float v) { return __float_as_uint(v) << 1; }
constexpr uint32_t kInfinite = 0xff000000u;
// 2^-90: below it the parts of a split value may be missing (see the top of the file)
constexpr uint32_t kSplitsFrom = (uint32_t)(127 - 90) << 24;

// Rows of 16 * PP bytes lie in LDS one behind the other; position p of row r holds piece p ^ row_swizzle<PP>(r), so that 16
// lanes that read one logical piece of 16 rows touch distinct banks (256 bytes of them).
template <int PP>
__device__ __forceinline__ int row_swizzle(int r) {
    static_assert((PP & (PP - 1)) == 0 && PP <= 16, "");
    return (r / (16 / PP)) & (PP - 1);
}

// A wave's weight fragment of one step: READS 16-byte (int8: 8-byte) LDS reads of a row, PARTS bf16 operands out of CHUNKS
// turns of conversion.
template <typename WT>
struct Weights;
template <>
struct Weights<float> {
    static constexpr int PARTS = 3, PIECE = 4, READS = 2, CHUNKS = 4, COST = 11;
    float v[8];
    __device__ __forceinline__ void read(int i, const unsigned char* row, int step, int half, int sw) {
        const float4 q = *reinterpret_cast<const float4*>(row + 16 * ((4 * step + 2 * half + i) ^ sw));
        v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
    }
    __device__ __forceinline__ void convert(int i, uint32_t (&o)[3][4]) const { split2(v[2 * i], v[2 * i + 1], o[0][i], o[1][i], o[2][i]); }
};
template <>
struct Weights<bf16_t> {
    static constexpr int PARTS = 1, PIECE = 8, READS = 1, CHUNKS = 1, COST = 0;
    uint4 v;
    __device__ __forceinline__ void read(int, const unsigned char* row, int step, int half, int sw) {
        v = *reinterpret_cast<const uint4*>(row + 16 * ((2 * step + half) ^ sw));
    }
    __device__ __forceinline__ void convert(int, uint32_t (&o)[1][4]) const { o[0][0] = v.x; o[0][1] = v.y; o[0][2] = v.z; o[0][3] = v.w; }
};
template <>
struct Weights<int8_t> {
    static constexpr int PARTS = 1, PIECE = 16, READS = 1, CHUNKS = 2, COST = 6;
    uint2 v;
    __device__ __forceinline__ void read(int, const unsigned char* row, int step, int half, int sw) {
        v = *reinterpret_cast<const uint2*>(row + 16 * (step ^ sw) + 8 * half);
    }
    __device__ __forceinline__ void convert(int i, uint32_t (&o)[1][4]) const {
        const uint32_t q = i ? v.y : v.x;
        o[0][2 * i] = widen2(q, 0);
        o[0][2 * i + 1] = widen2(q, 16);
    }
};
__device__ __forceinline__ float weight_value(float v) { return v; }
__device__ __forceinline__ float weight_value(bf16_t v) { return to_f32(v); }
__device__ __forceinline__ float weight_value(int8_t v) { return (float)v; }

// Columns c .. c + 3 of a row of K, in f32.  WHOLE: rows of whole 16-byte pieces on 16-byte boundaries; otherwise columns past
// the end count as zero.
template <bool WHOLE, typename T>
__device__ __forceinline__ void load4_f32(const T* row, int c, int K, float (&v)[4]) {
    struct __attribute__((aligned(4 * sizeof(T)))) Four {
        T v[4];
    };
    if constexpr (WHOLE) {
        const Four f = *reinterpret_cast<const Four*>(row + c);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = weight_value(f.v[i]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float w = weight_value(row[min(c + i, K - 1)]);
            v[i] = c + i < K ? w : 0.0f;
        }
    }
}

// A second, dense group in the same launch (the shared expert); rows 0: none.
template <typename WT>
struct F32Dense {
    const float* a;
    const WT* w;
    const float* scales;
    int N, K, rows;
    float *out, *gu_out;
};

// `parts`: GroupedArgs::parts (DMA, plain launches; otherwise 1).
// `sub`: this kernel's tiles in one of the tile table's, 1 or 2.  TB = blocks of 32 token rows per workgroup; FW = waves along the features (the workgroup owns 32 FW of them, or with
// SWIGLU as many gate and up rows each), STEPS = steps of 16 reduction columns a wave takes of a slice.  DMA: rows of whole
// 16-byte pieces on 16-byte boundaries and whole slices; otherwise both operands travel element by element.
template <typename WT, bool SWIGLU, int NW, int TB, int FW, int STEPS, bool DMA>
__global__ __launch_bounds__(NW * 64, 2) void grouped_f32_kernel(
    const float* __restrict__ a, const int* __restrict__ row_index, const WT* __restrict__ w, size_t w_expert_stride,
    const float* __restrict__ scales, size_t s_expert_stride, int N, int K, const int* __restrict__ tile_expert,
    const int* __restrict__ tile_row0, const int* __restrict__ tile_rows, const int* __restrict__ ntiles, int sub, int dense_rows,
    float* __restrict__ out, float* __restrict__ gu_out, const float* __restrict__ bw_gu, F32Dense<WT> g2, RoutedSlots slots,
    int parts, int part_rows) {
    typedef Weights<WT> W;
    constexpr int NTH = NW * 64;
    constexpr int KG = NW / FW;                   // wave groups that share out a slice's steps
    constexpr int FN = 32 * FW;
    constexpr int NB = SWIGLU ? 2 : 1;            // blocks of 32 weight rows a wave: gate and up, or plain
    constexpr int WR = NB * FN;                   // weight rows staged per slice
    constexpr int BM = 32 * TB;
    constexpr int SK = 16 * STEPS * KG;           // reduction columns of a slice
    constexpr int WROW = SK * (int)sizeof(WT), WPP = WROW / 16, TPP = SK / 8;  // pieces of a weight row, of a row of a plane
    constexpr int WSTAGE = WR * WROW, PLANE = BM * SK * 2, PBUF = 3 * PLANE;
    constexpr int WINST = WSTAGE / 1024;          // LDS-DMA instructions of a slice
    constexpr int DW = (WINST + NW - 1) / NW;     // ... a wave (waves left without one repeat another's)
    constexpr int TPIECES = BM * SK / 4;          // 16-byte pieces of raw token rows of a slice
    constexpr int NT = (TPIECES + NTH - 1) / NTH; // ... a thread (threads left without one repeat another's)
    constexpr int LOOP_BYTES = RING * WSTAGE + 2 * PBUF, MEET_BYTES = KG > 1 ? NW * NB * TB * 16 * 64 * 4 : 0;
    constexpr int USED_BYTES = LOOP_BYTES > MEET_BYTES ? LOOP_BYTES : MEET_BYTES;
    constexpr int LDS_BYTES = !SWIGLU || USED_BYTES > (int)sizeof(SlotsLds) ? USED_BYTES : (int)sizeof(SlotsLds);
    __shared__ __attribute__((aligned(16))) unsigned char lds[LDS_BYTES];
    __shared__ int own_token[SWIGLU ? 2 * kSlotsTileM : 1];  // (read once more behind the loop)
    __shared__ uint32_t row_top[BM];                         // the rows' largest magnitudes
    unsigned char* const planes = lds + RING * WSTAGE;

    // ---- which tile: each XCD (workgroup number mod 8) walks a contiguous range of tiles with one expert's row tiles
    // innermost, so that a weight slice is fetched by one L2
    // (without tables: what the router left behind, see RoutedSlots; the second group's tiles come behind the routed ones)
    const bool own = SWIGLU && slots.expert_of != nullptr;  // uniform over the launch
    SlotsLds& sl = *reinterpret_cast<SlotsLds*>(lds);
    RoutedCounts rc{};
    if (own) {
        if (blockIdx.x == gridDim.x - 1) return routed_rest(slots, lds);
        rc = routed_counts<NTH>(slots, sl);
    }
    int tiles_n = (N + FN - 1) / FN;
    int tiles_m = dense_rows >= 0 ? (dense_rows + BM - 1) / BM : (own ? rc.ntiles : *ntiles) * sub;
    const int total1 = tiles_m * tiles_n;
    const int tiles_n2 = (g2.N + FN - 1) / FN, tiles_m2 = (g2.rows + BM - 1) / BM;
    const int whole = total1 + tiles_m2 * tiles_n2, total = SWIGLU ? whole : whole * parts;
    const int per_xcd = (total + 7) / 8;
    const int local = blockIdx.x >> 3;
    if (local >= per_xcd) return;
    int pid = (blockIdx.x & 7) * per_xcd + local;
    if (pid >= total) return;
    const int part = SWIGLU || parts == 1 ? 0 : pid / whole;  // (uniform over the workgroup, like all of this)
    pid -= part * whole;
    const bool second = pid >= total1;
    if (second) {  // (uniform over the workgroup)
        pid -= total1;
        tiles_n = tiles_n2;
        tiles_m = tiles_m2;
        a = g2.a;
        row_index = nullptr;
        w = g2.w;
        scales = g2.scales;
        N = g2.N;
        K = g2.K;
        dense_rows = g2.rows;
        out = g2.out;
        gu_out = g2.gu_out;
        part_rows = g2.rows;
    }
    const int pitch = K;  // of the rows of both operands
    if (DMA && !SWIGLU && parts > 1) {  // this workgroup's slices
        const int from = K / SK * part / parts * SK, to = K / SK * (part + 1) / parts * SK;
        a += from;
        w += from;
        K = to - from;
        out += (size_t)part * part_rows * N;
    }
    constexpr int GROUP_M = 8;
    const int per_group = GROUP_M * tiles_n;
    const int first_m = pid / per_group * GROUP_M;
    const int gsize = min(GROUP_M, tiles_m - first_m);
    const int in_g = pid % per_group;
    const int tm_idx = first_m + in_g % gsize;
    const int n0 = in_g / gsize * FN;

    int expert, row0, rows, skip = 0;
    if (dense_rows >= 0) {
        expert = 0;
        row0 = tm_idx * BM;
        rows = min(BM, dense_rows - row0);
    } else {
        const int entry = sub == 2 ? tm_idx >> 1 : tm_idx;
        skip = sub == 2 ? (tm_idx & 1) * BM : 0;
        if (own) {
            const RoutedTile t = routed_tile<NTH>(slots, rc, entry, n0 == 0 && skip == 0, sl, own_token);
            expert = t.expert;
            row0 = t.row0 + skip;
            rows = min(BM, t.rows - skip);
        } else {
            expert = tile_expert[entry];
            row0 = tile_row0[entry] + skip;
            rows = min(BM, tile_rows[entry] - skip);
        }
        if (rows <= 0) return;
    }
    const bool own_rows = own && !second;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fw = wv % FW, grp = wv / FW;    // which 32 features; which steps of every slice
    const int lr = lane & 31, lh = lane >> 5;
    const WT* const wbase = w + (size_t)expert * w_expert_stride;
    // (rows past the end of the group, features past N: any valid one, products never stored)
    auto token_row = [&](int r) {
        const int rr = r < rows ? r : 0;
        return a + (size_t)(own_rows ? own_token[skip + rr] : row_index ? row_index[row0 + rr] : row0 + rr) * pitch;
    };
    auto weight_row = [&](int q) {  // q < FN: gate (or plain) feature n0 + q; q >= FN: the matching up row
        const int feat = n0 + (q % FN);
        const int fr = feat < N ? feat : 0;
        return wbase + (size_t)((SWIGLU && q >= FN) ? N + fr : fr) * pitch;
    };

    // ---- staging
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    const WT* wsrc[DMA ? DW : 1];
    const float* tsrc[NT];
    int tcol[NT];
    unsigned char* tdst[NT];
    float top[NT];  // the largest value so far of the row of piece i, signs aside (NaN: there is one)
    auto piece_row = [&](int i) { return (i * NTH + tid) % TPIECES / (SK / 4); };
    constexpr int NWE = DMA ? 1 : WR * SK / NTH;
    WT pend_w[NWE];
    u32x4 pend_t[2][NT];  // raw row values of two slices under way
    if constexpr (DMA) {
#pragma unroll
        for (int i = 0; i < DW; ++i) {
            const int p = ((wv * DW + i) % WINST) * 64 + lane, r = p / WPP;
            wsrc[i] = weight_row(r) + W::PIECE * ((p % WPP) ^ row_swizzle<WPP>(r));
        }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int r = piece_row(i), c = (i * NTH + tid) % (SK / 4);
        top[i] = 0.0f;
        tsrc[i] = token_row(r);
        tcol[i] = 4 * c;
        tdst[i] = planes + r * (SK * 2) + 16 * ((c >> 1) ^ row_swizzle<TPP>(r)) + 8 * (c & 1);
    }
    const int KT = (K + SK - 1) / SK;
    // (slices past the last only keep the wait counts: fetched again and never read)
    auto dma_w = [&](int i, int kt, int slot) {
        f32_issue_dma(lds0 + (uint32_t)(slot * WSTAGE + ((wv * DW + i) % WINST) * 1024), wsrc[i] + min(kt, KT - 1) * SK);
    };
    auto load_t = [&](int i, int kt, u32x4& to) {
        if constexpr (DMA) {
            f32_issue_load(to, tsrc[i] + min(kt, KT - 1) * SK + tcol[i]);
        } else {
            const int c = kt * SK + tcol[i];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float v = tsrc[i][min(c + q, K - 1)];
                to[q] = c + q < K ? __float_as_uint(v) : 0u;  // (columns past the end of a row count as zero)
            }
        }
    };
    auto load_w = [&](int kt) {
        if constexpr (!DMA) {
#pragma unroll
            for (int i = 0; i < NWE; ++i) {
                const int e = i * NTH + tid;
                pend_w[i] = weight_row(e / SK)[min(kt * SK + e % SK, K - 1)];
            }
        }
    };
    auto put_w = [&](int slot) {
        if constexpr (!DMA) {
#pragma unroll
            for (int i = 0; i < NWE; ++i) {
                const int e = i * NTH + tid, r = e / SK, c = e % SK;
                reinterpret_cast<WT*>(lds + slot * WSTAGE + r * WROW + 16 * ((c / W::PIECE) ^ row_swizzle<WPP>(r)))[c % W::PIECE] = pend_w[i];
            }
        }
    };
    // the rows' planes: [buffer][plane][row][SK / 8 pieces of 8 bf16]
    uint32_t cv[3][2];
    auto split_t = [&](int i, int half, const u32x4& v) {
        const float x = __uint_as_float(half ? v.z : v.x), y = __uint_as_float(half ? v.w : v.y);
        top[i] = __builtin_elementwise_maximum(__builtin_elementwise_maximum(top[i], __builtin_fabsf(x)), __builtin_fabsf(y));
        split2(x, y, cv[0][half], cv[1][half], cv[2][half]);
    };
    auto put_t = [&](int i, int buf) {
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(tdst[i] + buf * PBUF + p * PLANE) = make_uint2(cv[p][0], cv[p][1]);
    };

    // Six terms a step are six roundings of a sum where the f32 unit has eight; the five small ones are therefore summed
    // apart, where a rounding is 2^-8 of one of the large sum's, unless the wave groups share out the steps anyway.
    constexpr bool APART = W::PARTS == 3 && KG == 1;
    floatx16 acc[NB][TB], low[NB][TB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[nb][t][v] = low[nb][t][v] = 0.0f;

    // ---- fragments of one step
    struct Operands {
        uint4 t[TB][3];
        uint32_t w[NB][W::PARTS][4];
    };
    W wraw[NB];
    const int wsw = row_swizzle<WPP>(lr), tsw = row_swizzle<TPP>(lr);  // (32 rows on, the same)
    const unsigned char* const wrow = lds + (fw * 32 + lr) * WROW;
    const unsigned char* const trow = planes + lr * (SK * 2);
    auto read_t = [&](Operands& o, int i, int buf, int s) {
        const int t = i / 3, p = i % 3;
        o.t[t][p] = *reinterpret_cast<const uint4*>(trow + buf * PBUF + p * PLANE + t * (32 * SK * 2) + 16 * ((2 * (grp * STEPS + s) + lh) ^ tsw));
    };
    auto read_w = [&](int i, int slot, int s) {
        const int nb = i / W::READS;
        wraw[nb].read(i % W::READS, wrow + slot * WSTAGE + nb * (FN * WROW), grp * STEPS + s, lh, wsw);
    };
    // term number i of a product, the smallest first: which part of the weight, which of the row
    constexpr int TERMS = W::PARTS == 3 ? 6 : 3;
    auto multiply = [&](auto m_tag, const Operands& o) {
        constexpr int m = decltype(m_tag)::value, term = m / (NB * TB), nb = m / TB % NB, t = m % TB;
        constexpr int wp = W::PARTS == 3 ? (term == 0 ? 2 : (term == 1 || term == 3) ? 1 : 0) : 0;
        constexpr int tp = W::PARTS == 3 ? (term == 2 ? 2 : (term == 1 || term == 4) ? 1 : 0) : 2 - term;
        const uint4 wf = make_uint4(o.w[nb][wp][0], o.w[nb][wp][1], o.w[nb][wp][2], o.w[nb][wp][3]);
        floatx16& sum = APART && term < TERMS - 1 ? low[nb][t] : acc[nb][t];
        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wf), __builtin_bit_cast(bf16x8, o.t[t][tp]), sum, 0, 0, 0);
    };

    // ---- one step: its multiplies with everything else between them, each piece behind a multiply of its own (the order is
    // pinned): the reads of the next step's fragments; with FETCH the weights of slice kt + 3 under way; with CONV the rows
    // of slice `ck` from registers to their planes and those of slice ck + 2 under way; the split of the next step's weights
    auto step = [&](auto fetch_tag, auto conv_tag, const Operands& cur, Operands& nxt, int rslot, int rbuf, int rs, int kt,
                    int fslot, int ck, u32x4 (&set)[NT]) {
        constexpr bool FETCH = decltype(fetch_tag)::value, CONV = decltype(conv_tag)::value;
        constexpr int NM = NB * TB * TERMS;
        constexpr int RW = NB * W::READS, RT = 3 * TB, F = FETCH && DMA ? DW : 0, C = CONV ? 3 * NT : 0, X = NB * W::CHUNKS;
        constexpr int OPS = RW + RT + F + C + X;
        constexpr int COST = RW + RT + 4 * F + 10 * C + W::COST * X;
        auto before = [](int i) constexpr {  // cost of what comes in front of operation i
            int c = 0;
            for (int j = 0; j < i; ++j)
                c += j < RW + RT ? 1 : j < RW + RT + F ? 4 : j < RW + RT + F + C ? 10 : W::COST;
            return c;
        };
        auto op = [&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value;
            if constexpr (i < RW) {
                read_w(i, rslot, rs);
            } else if constexpr (i < RW + RT) {
                read_t(nxt, i - RW, rbuf, rs);
            } else if constexpr (i < RW + RT + F) {
                dma_w(i - RW - RT, kt + 3, fslot);
            } else if constexpr (i < RW + RT + F + C) {
                constexpr int j = i - RW - RT - F, u = j / 3;
                if constexpr (j % 3 < 2) {
                    split_t(u, j % 3, set[u]);
                } else {
                    put_t(u, ck & 1);
                    load_t(u, ck + 2, set[u]);
                }
            } else {
                constexpr int j = i - RW - RT - F - C;
                wraw[j / W::CHUNKS].convert(j % W::CHUNKS, nxt.w[j / W::CHUNKS]);
            }
        };
        if constexpr (FETCH && !DMA) {
            put_w(fslot == 0 ? 2 : fslot - 1);  // slice kt + 2
            load_w(kt + 3);
        }
        f32_for<0, NM>([&](auto m_tag) {
            constexpr int m = decltype(m_tag)::value;
            multiply(m_tag, cur);
            __builtin_amdgcn_sched_barrier(0);
            f32_for<0, OPS>([&](auto i_tag) {
                constexpr int at = COST == 0 ? 0 : before(decltype(i_tag)::value) * NM / (COST + 1);
                if constexpr (at == m) op(i_tag);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    // ---- pipeline.  The barrier of a slice stands in front of its last step: by then every wave has read all of the slice's
    // fragments, and behind it the next slice is complete in LDS.  Loads retire in order: of what was issued since the last
    // barrier nothing need have landed, of what was issued before that all must (weights of the next slice, row values of
    // the next conversion).
    constexpr bool ONE = STEPS == 1;
    // Everything that the first slices need is requested at once: the rows of slices 0 and 1 (or 0 alone) in registers of
    // their own, those of the next two where the loop takes them from - set p holds the slice that the conversions in the
    // slices of parity p (or, with two steps, of the other parity) take next.
    u32x4 first[2][NT];
    f32_for<0, NT>([&](auto i) { load_t(i, 0, first[0][i]); });
    if constexpr (ONE) f32_for<0, NT>([&](auto i) { load_t(i, 1, first[1][i]); });
    auto first_w = [&](int k) {
        if constexpr (DMA) {
#pragma unroll
            for (int i = 0; i < DW; ++i) dma_w(i, k, k);
        } else {
            load_w(k);
            if (k < 2) put_w(k);
        }
    };
    first_w(0);
    f32_for<0, NT>([&](auto i) { load_t(i, 2, pend_t[0][i]); });
    f32_for<0, NT>([&](auto i) { load_t(i, ONE ? 3 : 1, pend_t[1][i]); });
    first_w(1);
    first_w(2);
    if (tid < BM) row_top[tid] = 0;  // (every wave passes a barrier before it is read)
    auto wait = [&](auto n_tag) {
#pragma unroll
        for (int i = 0; i < NT; ++i) asm volatile("" : "+v"(pend_t[0][i]), "+v"(pend_t[1][i]));
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(decltype(n_tag)::value) : "memory");
#pragma unroll
        for (int i = 0; i < NT; ++i) asm volatile("" : "+v"(pend_t[0][i]), "+v"(pend_t[1][i]));
    };
    typedef std::integral_constant<int, 0> All;
    typedef std::integral_constant<int, DMA ? DW + NT : 63> Older;
    wait(std::integral_constant<int, DMA ? 2 * NT + 2 * DW : 63>{});
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        asm volatile("" : "+v"(first[0][i]));
        if constexpr (ONE) asm volatile("" : "+v"(first[1][i]));
    }
    auto convert_now = [&](int buf) {
        f32_for<0, NT>([&](auto i) {
            split_t(i, 0, first[buf][i]);
            split_t(i, 1, first[buf][i]);
            put_t(i, buf);
        });
    };
    convert_now(0);
    if constexpr (ONE) convert_now(1);
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    Operands oa, ob;
    f32_for<0, NB * W::READS>([&](auto i) { read_w(i, 0, 0); });
    f32_for<0, 3 * TB>([&](auto i) { read_t(oa, i, 0, 0); });
    f32_for<0, NB * W::CHUNKS>([&](auto i) { wraw[i / W::CHUNKS].convert(i % W::CHUNKS, oa.w[i / W::CHUNKS]); });
    wait(All{});
    int s0 = 0;  // kt % RING
    typedef std::true_type Yes;
    typedef std::false_type No;
    auto slice = [&](int kt, auto par_tag, Operands& c, Operands& n) {
        constexpr int par = decltype(par_tag)::value;  // kt % 2
        const int s1 = s0 == 2 ? 0 : s0 + 1;
        if constexpr (ONE) {
            wait(Older{});
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            step(Yes{}, Yes{}, c, n, s1, par ^ 1, 0, kt, s0, kt + 2, pend_t[par]);
        } else {
            static_assert(STEPS <= 2, "one step in front of the barrier");
            step(No{}, Yes{}, c, n, s0, par, 1, kt, 0, kt + 1, pend_t[par ^ 1]);
            wait(Older{});
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            step(Yes{}, No{}, n, c, s1, par ^ 1, 0, kt, s0, 0, pend_t[0]);
        }
        s0 = s1;
    };
    typedef std::integral_constant<int, 0> Even;
    typedef std::integral_constant<int, 1> Odd;
    int kt = 0;
    for (; kt + 2 <= KT; kt += 2) {
        slice(kt, Even{}, oa, ob);
        if constexpr (ONE) slice(kt + 1, Odd{}, ob, oa);
        else slice(kt + 1, Odd{}, oa, ob);
    }
    if (kt < KT) slice(kt, Even{}, oa, ob);
    wait(All{});  // the LDS is used again below, and nothing may land after the workgroup has ended
#pragma unroll
    for (int i = 0; i < NT; ++i) atomicMax(&row_top[piece_row(i)], magnitude(top[i]));
    __syncthreads();

    // ---- wave groups that share out the reduction meet in LDS: group g finishes quads (four values) g OQ .. + OQ - 1 of the
    // wave's TB * 4, the groups' shares summed in their order
    constexpr int OQ = TB * 4 / KG;
    float mine[NB][OQ][4];
    if constexpr (KG > 1) {
        float4* const ex = reinterpret_cast<float4*>(lds);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int q = 0; q < TB * 4; ++q) {
                const floatx16& v = acc[nb][q / 4];
                ex[((wv * NB + nb) * (TB * 4) + q) * 64 + lane] =
                    make_float4(v[4 * (q % 4)], v[4 * (q % 4) + 1], v[4 * (q % 4) + 2], v[4 * (q % 4) + 3]);
            }
        __syncthreads();
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int q = 0; q < OQ; ++q) {
                float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
                for (int g = 0; g < KG; ++g) {
                    const float4 v = ex[(((g * FW + fw) * NB + nb) * (TB * 4) + grp * OQ + q) * 64 + lane];
                    sum.x += v.x;
                    sum.y += v.y;
                    sum.z += v.z;
                    sum.w += v.w;
                }
                mine[nb][q][0] = sum.x; mine[nb][q][1] = sum.y; mine[nb][q][2] = sum.z; mine[nb][q][3] = sum.w;
            }
    } else {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int q = 0; q < OQ; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = acc[nb][q / 4][4 * (q % 4) + i];
                    mine[nb][q][i] = APART ? v + low[nb][q / 4][4 * (q % 4) + i] : v;
                }
    }

    // Accumulator element v of lane l: feature 8 (v / 4) + 4 (l / 32) + v % 4 of the wave's block, token l % 32.
    // finish: four features from `f` on of one row of the layer's tables, what becomes of the sums
    auto finish = [&](auto whole_tag, size_t orow, int f, float (&g)[4], float (&u)[4]) {
        constexpr bool WHOLE = decltype(whole_tag)::value;  // N a multiple of 4: in or out as a whole, on 16-byte boundaries
        const int n = N - f;
        auto store4 = [&](float* to, const float (&v)[4]) {
            if constexpr (WHOLE) {
                *reinterpret_cast<float4*>(to) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (i < n) to[i] = v[i];
            }
        };
        if constexpr (sizeof(WT) == 1) {
            const float* const sc = scales + (size_t)expert * s_expert_stride;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int fi = min(f + i, N - 1);
                g[i] *= sc[fi];
                if constexpr (SWIGLU) u[i] *= sc[N + fi];
            }
        }
        float y[4];
        if constexpr (SWIGLU) {
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = silu_f32(g[i]) * u[i];
            if (gu_out != nullptr) {  // uniform: the pre-activations G | U [rows, 2 N] kept for a backward pass
                float* const grow = gu_out + orow * 2 * N + f;
                store4(grow, g);
                store4(grow + N, u);
            }
        } else if (bw_gu != nullptr) {  // uniform
            // SwiGlu::backward (src/ffn.rs:87-120) on the way out: the product row is the gradient of the
            // hidden row; dG = dH * U * silu'(G), dU = dH * silu(G) go to `gu_out`, `out` is not written.
            const size_t off = orow * 2 * N + f;
            float gv[4], uv[4], dg[4], du[4];
            if constexpr (WHOLE) {
                const float4 g4 = *reinterpret_cast<const float4*>(bw_gu + off), u4 = *reinterpret_cast<const float4*>(bw_gu + off + N);
                gv[0] = g4.x; gv[1] = g4.y; gv[2] = g4.z; gv[3] = g4.w;
                uv[0] = u4.x; uv[1] = u4.y; uv[2] = u4.z; uv[3] = u4.w;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    gv[i] = bw_gu[off + min(i, n - 1)];
                    uv[i] = bw_gu[off + N + min(i, n - 1)];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float sg = 1.0f / (1.0f + __expf(-gv[i]));
                dg[i] = g[i] * uv[i] * (sg * (1.0f + gv[i] * (1.0f - sg)));  // silu', src/ffn.rs:235-238
                du[i] = g[i] * (gv[i] * sg);
            }
            store4(gu_out + off, dg);
            store4(gu_out + off + N, du);
            return;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = g[i];
        }
        store4(out + orow * N + f, y);
    };
    auto token_of = [&](int q) { return (grp * OQ + q) / 4 * 32 + lr; };
    auto feature_of = [&](int q) { return n0 + fw * 32 + 8 * ((grp * OQ + q) % 4) + 4 * lh; };
    // An infinity (or a value within a rounding of the largest) splits into parts that cancel or meet a zero part of the other
    // operand: the sum is then not a number where the product of the values themselves may well be one.  And a product of two
    // first parts may be larger than that of the values by 2^-7, and past the largest f32 where that is not.  At the other end
    // parts are missing (see the top of the file).  Taken again from the values, by the f32 matrix unit, the whole wave block
    // at once and straight from memory, are therefore sums that are not finite, those of rows with a NaN in them aside; sums
    // below 2^-90 that are not zero; and all sums of a row whose largest value is below 2^-90 and not zero.  Only they take
    // the new sums: what a row comes out as does not depend on its neighbours.  us a forward, 1024 rows, d 512, 8 experts of
    // 1408 in f32, plain rows 93 (92.5 without a look at small values): a row of NaN among them 94, all NaN 86, all infinite
    // 156; one lane after the other 1231, 2935 and 2934, and 126, 115 and 115 with every product on the f32 unit.  8 experts of
    // 352 and a shared one, bf16 weights, plain 41: 41, 40 and 103.
    // (the whole lane at once first: hardly ever is there more to find out)
    float most = 0.0f, least = HUGE_VALF;
    bool tiny = false;
#pragma unroll
    for (int q = 0; q < OQ; ++q) {
        tiny = tiny || row_top[token_of(q)] - 1 < kSplitsFrom - 1;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                most = __builtin_elementwise_maximum(most, __builtin_fabsf(mine[nb][q][i]));
                least = __builtin_elementwise_minimum(least, __builtin_fabsf(mine[nb][q][i]));
            }
    }
    uint32_t odd = 0;  // quads to take again
    if (__ballot(tiny || !(most < HUGE_VALF && least >= 0x1p-90f)) != 0ull) {
#pragma unroll
        for (int q = 0; q < OQ; ++q) {
            const uint32_t largest = row_top[token_of(q)];
            if (token_of(q) >= rows || feature_of(q) >= N || largest > kInfinite) continue;
            bool again = largest - 1 < kSplitsFrom - 1;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t m = magnitude(mine[nb][q][i]);
                    again = again || m >= kInfinite || m - 1 < kSplitsFrom - 1;
                }
            if (again) odd |= 1u << q;
        }
    }
    if (__ballot(odd != 0) != 0ull) {
        constexpr int OT = OQ >= 4 ? OQ / 4 : 1;  // blocks of 32 rows that this wave finishes
        const float* tr[OT];
        const WT* wr[NB];
        floatx16 sum[NB][OT];
#pragma unroll
        for (int t = 0; t < OT; ++t) tr[t] = token_row((grp * OQ / 4 + t) * 32 + lr);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            wr[nb] = weight_row(nb * FN + fw * 32 + lr);
#pragma unroll
            for (int t = 0; t < OT; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) sum[nb][t][v] = 0.0f;
        }
        // multiply j of a step takes column 4 (l / 32) + j of lane l in both operands
#pragma unroll 1
        for (int c0 = 0; c0 < K; c0 += 32) {
            float tv[4][OT][4], wv4[4][NB][4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = c0 + 8 * u + 4 * lh;
#pragma unroll
                for (int t = 0; t < OT; ++t) load4_f32<DMA>(tr[t], c, K, tv[u][t]);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) load4_f32<DMA>(wr[nb], c, K, wv4[u][nb]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                        for (int t = 0; t < OT; ++t)
                            sum[nb][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv4[u][nb][j], tv[u][t][j], sum[nb][t], 0, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < OQ; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {  // (which quad of its block q is, is known at compile time where the wave has whole blocks)
                if (!((odd >> q) & 1) || v != (grp * OQ + q) % 4) continue;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int i = 0; i < 4; ++i) mine[nb][q][i] = sum[nb][OQ >= 4 ? q / 4 : 0][4 * v + i];
            }
    }
    auto store_tile = [&](auto whole_tag) {
#pragma unroll
        for (int q = 0; q < OQ; ++q) {
            const int tok = token_of(q), f = feature_of(q);
            if (tok >= rows || f >= N) continue;
            float g[4], u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                g[i] = mine[0][q][i];
                u[i] = mine[NB - 1][q][i];
            }
            finish(whole_tag, (size_t)(row0 + tok), f, g, u);
        }
    };
    if (N % 4 == 0) store_tile(Yes{});
    else store_tile(No{});
}

}  // namespace

int f32_tile_m(int rows, int groups) { return rows <= 32 * groups ? 32 : 64; }

// What the f32 matrix-core kernel set asks for: whole slices of the reduction, whole pieces of an output row
bool f32_shape_ok(int N, int K) { return K % 32 == 0 && K >= 32 && N % 4 == 0 && N >= 4; }

// Tokens x features of a workgroup, and its waves.  A launch is bound by the length of one workgroup's chain until there
// are about as many workgroups as compute units, and by the multiplies from there on, which the larger tiles feed best.
// So: the smallest tile of which there is at most one a compute unit (bf16 and int8 weights, a third of the multiplies
// and of the LDS a tile: some more of them together), then 64 x 128.  us, all at 8 experts top-2, d 512 (swept before
// the rows' largest values were looked at: the large ones take 1 % more now, whichever the tile):
//   f32, gate/up of 1408     32x32 / 32x64 / 64x64 / 64x128 / the same on eight waves: 1 token 9.8 / 13.3 / 17.2 / 25.8 / -, 8
//     tokens 14.0 / 12.7 / 17.6 / 26.2 / -, 128 20.2 / 19.7 / 17.6 / 25.8 / 23.9, 256 30.1 / 27.5 / 27.6 / 27.9 / 25.4, 1024
//     71.1 / 59.6 / 52.9 / 46.4 / 50.1, 8192 499 / 374 / 301 / 284 / 319
//   f32, down from 1408      128 tokens 13.0 / 17.0 / 22.8 / 34.6 / 29.6, 256 18.8 / 17.2 / 23.4 / 33.8 / 29.9, 512 24.3 / 25.4
//     / 23.3 / 34.4 / 30.2, 1024 39.6 / 35.4 / 36.6 / 34.8 / 31.5, 8192 242 / 192 / 167 / 159 / 175
//   bf16, gate/up of 682     32 tokens 8.9 / 8.5 / 11.6 / 14.5, 256 12.7 / 11.9 / 13.1 / 16.4, 1024 24.4 / 20.7 / 19.6 / 19.6,
//     2048 40.7 / 32.0 / 31.2 / 29.4
// A last feature tile that is mostly empty costs more than half as wide tiles do: 64 experts of 704 (five and a half tiles
// of 128), d 1024, 2048 tokens, six a row: 268 us in 64x128, 248 in 64x64.
static long long f32_tiles(const GroupedArgs& g, int rows, int features) {
    const int S = g.dense_rows >= 0 ? g.dense_rows : g.routed_rows, E = g.dense_rows >= 0 ? 1 : g.groups;
    // tiles of a group's rows: a last one half full, or one tile for each group that gets any
    const int hit = std::min(E, S);
    return (long long)std::max(S / rows + (hit + 1) / 2, hit) * ((g.N + features - 1) / features) +
           (long long)((g.dense2.rows + rows - 1) / rows) * ((g.dense2.N + features - 1) / features);
}
enum class F32Tile { T32x32, T32x64, T64x64, T64x128, T64x128x8 };
static F32Tile f32_tile(const GroupedArgs& g, bool f32_weights, bool small_slices) {
    auto tiles = [&](int rows, int features) { return f32_tiles(g, rows, features); };
    if (tiles(32, 32) <= 256 && small_slices) return F32Tile::T32x32;
    if (tiles(32, 64) <= (f32_weights ? 256 : 600) || (g.dense_rows < 0 && g.tile_m == 32)) return F32Tile::T32x64;
    if (tiles(64, 64) <= 256) return F32Tile::T64x64;
    if (f32_weights && tiles(64, 128) <= 256) return F32Tile::T64x128x8;
    return (g.N + 127) / 128 * 128 * 20 > (g.N + 63) / 64 * 64 * 21 ? F32Tile::T64x64 : F32Tile::T64x128;
}

struct F32Plan {
    F32Tile tile;
    bool aligned;
    int workgroups;  // about as many
};
static F32Plan f32_plan(const GroupedArgs& g, int weight_size) {
    auto whole = [](const void* p, size_t pitch) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && pitch % 16 == 0; };
    auto group = [&](const void* a, const void* w, int K) { return K % 32 == 0 && whole(a, (size_t)K * 4) && whole(w, (size_t)K * weight_size); };
    const GroupedArgs::Dense& d2 = g.dense2;
    const bool f32 = weight_size == 4;
    F32Plan p;
    p.aligned = group(g.a, g.w, g.K) && g.w_expert_stride * weight_size % 16 == 0 && (d2.rows == 0 || group(d2.a, d2.w, d2.K));
    p.tile = f32_tile(g, f32, !p.aligned || (g.K % 64 == 0 && d2.K % 64 == 0));
    if (f32 && !p.aligned && (p.tile == F32Tile::T64x128 || p.tile == F32Tile::T64x128x8)) p.tile = F32Tile::T64x64;
    const int rows = p.tile == F32Tile::T32x32 || p.tile == F32Tile::T32x64 ? 32 : 64;
    const int features = p.tile == F32Tile::T32x32 ? 32 : p.tile == F32Tile::T32x64 || p.tile == F32Tile::T64x64 ? 64 : 128;
    p.workgroups = (int)std::min<long long>(f32_tiles(g, rows, features), 1 << 30);
    return p;
}

int f32_workgroups(const GroupedArgs& g, WeightKind wk) {
    return f32_plan(g, wk == WeightKind::F32 ? 4 : wk == WeightKind::BF16 ? 2 : 1).workgroups;
}

// A tile's chain of slices is what a small down launch waits for, so its reduction is shared out until there is a workgroup for
// every compute unit: in halves or quarters, whose sums the combine adds up.  us a forward, whole / 2 parts / 4 parts, f32 weights: d 512,
// 8 experts of 1408, 1 row (32 tiles) 32.8 / 29.2 / 28.0, 2 rows (64) 32.8 / 29.8 / 27.9, 8 rows (128) 36.6 / 33.2 / 33.8, 64 rows 37.7 /
// 35.0 / 35.5; d 256, 4 experts of 1408, all four a row, 20 rows (32) 32.5 / 29.1 / 28.1; d 768, 8 of 1408 and a shared one, 2 rows (120)
// 36.6 / 33.8 / 35.0, 16 rows (216) 42.4 / 42.8 / 44.2.  A second workgroup on some of the compute units takes back what the shorter
// chain gives: d 512, 8 of 1408, 1024 rows (144) 94.5 / 101.1 / 98.5.  Nor is there anything in a short one: of 700 shapes under those
// lines (d 64 to 1024, 4 to 32 experts of 96 to 2080, f32, bf16 and int8 weights, 1 to 500 rows) the ones of 96 to 160 columns are 0.7 % slower
// in parts on average, of 192 to 256 0.9 % faster and up to 6 % slower (d 256, 8 of 256 and a shared one, four a row, 65 rows 26.3 / 28.0 in
// quarters), of 352 4 % faster and 2 slower at most, of 2048 22.
// Errors against 64 bits become smaller (d 512, 8 of 1408, 1 row 4.0e-7 / 3.1e-7, 64 rows 4.7e-7 / 4.2e-7).  What is taken again (see
// `odd`) is so part by part: infinities and NaN meet in the combine's sum as they would in the whole one.
// Whole slices of every tile that either group may get, by itself too (a stage's replay): of 64 columns where the widths have them.
int f32_parts(const GroupedArgs& g, WeightKind wk) {
    const F32Plan p = f32_plan(g, wk == WeightKind::F32 ? 4 : wk == WeightKind::BF16 ? 2 : 1);
    const int K2 = g.dense2.rows > 0 ? g.dense2.K : g.K;
    if (!p.aligned || std::min(g.K, K2) < 288) return 1;
    auto slices = [](int K) { return K % 64 == 0 ? K / 64 : K / 32; };
    const int most = std::min(slices(g.K), slices(K2));
    int parts = 1;
    while (parts < 4 && 2 * parts * p.workgroups <= 256 && 2 * parts <= most) parts *= 2;
    return parts;
}

// Whole slices of both down products, or of neither: the routed experts' kernel stays the one they have by themselves.
bool f32_joins(int F, int Fs) { return F == Fs || (F % 64 == 0 && Fs % 64 == 0); }

template <typename WT>
static hipError_t launch_f32_t(const GroupedArgs& g, hipStream_t s) {
    if (g.dense_rows < 0 && g.tile_m != 32 && g.tile_m != 64) return hipErrorInvalidValue;
    if (g.slots.expert_of && (!g.swiglu || g.dense_rows >= 0 || g.slots.layout.tile_m != g.tile_m)) return hipErrorInvalidValue;
    if (g.dense2.rows > 0 && (g.dense_rows >= 0 || !g.dense2.gu_out != !g.gu_out || g.swiglu_grad_gu)) return hipErrorInvalidValue;
    constexpr bool F32 = sizeof(WT) == 4;
    const F32Plan plan = f32_plan(g, sizeof(WT));
    const bool aligned = plan.aligned;
    const GroupedArgs::Dense& d2 = g.dense2;
    const F32Dense<WT> g2{static_cast<const float*>(d2.a), static_cast<const WT*>(d2.w), d2.scales, d2.N, d2.K, d2.rows,
                          static_cast<float*>(d2.out), static_cast<float*>(d2.gu_out)};
    bool refused = false;
    auto go = [&](auto swiglu_tag, auto nw_tag, auto tb_tag, auto fw_tag, auto steps_tag) {
        constexpr bool SW = decltype(swiglu_tag)::value;
        constexpr int FW = decltype(fw_tag)::value, FN = 32 * FW, BM = 32 * decltype(tb_tag)::value;
        constexpr int NW = decltype(nw_tag)::value, STEPS = decltype(steps_tag)::value;
        const int tiles_m = g.dense_rows >= 0 ? (g.dense_rows + BM - 1) / BM : g.max_tiles * (g.tile_m / BM);
        const int total = ((g.N + FN - 1) / FN * tiles_m + (d2.N + FN - 1) / FN * ((d2.rows + BM - 1) / BM)) * g.parts;
        if (total <= 0) return;
        const int rest = SW && g.slots.expert_of ? 1 : 0;  // (routed_rest)
        const int sub = g.tile_m / BM;
        auto launch = [&](auto dma_tag) {
            RB_LAUNCH((grouped_f32_kernel<WT, SW, NW, BM / 32, FW, STEPS, decltype(dma_tag)::value>), dim3((total + 7) / 8 * 8 + rest),
                      dim3(64 * NW), 0, s, static_cast<const float*>(g.a), g.row_index, static_cast<const WT*>(g.w), g.w_expert_stride,
                      g.scales, g.s_expert_stride, g.N, g.K, g.tile_expert, g.tile_row0, g.tile_rows, g.ntiles, sub, g.dense_rows,
                      static_cast<float*>(g.out), static_cast<float*>(g.gu_out), static_cast<const float*>(g.swiglu_grad_gu), g2,
                      g.slots, g.parts, g.part_rows);
        };
        constexpr int SK = 16 * STEPS * (NW / FW);
        if (aligned && g.K % SK == 0 && d2.K % SK == 0) launch(std::true_type{});
        else if (g.parts > 1) refused = true;  // (f32_parts does not ask for it)
        else if constexpr (!(F32 && FW == 4)) launch(std::false_type{});  // (f32_tile does not ask for it)
    };
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, 2> Two;
    typedef std::integral_constant<int, 4> Four;
    typedef std::integral_constant<int, 8> Eight;
    auto pick = [&](auto swiglu_tag) {
        typedef std::integral_constant<int, decltype(swiglu_tag)::value && F32 ? 1 : 2> Steps;
        switch (plan.tile) {
            case F32Tile::T32x32: return go(swiglu_tag, Four{}, One{}, One{}, One{});
            case F32Tile::T32x64: return go(swiglu_tag, Four{}, One{}, Two{}, One{});
            case F32Tile::T64x64: return go(swiglu_tag, Four{}, Two{}, Two{}, One{});
            case F32Tile::T64x128: return go(swiglu_tag, Four{}, Two{}, Four{}, Steps{});
            case F32Tile::T64x128x8:
                if constexpr (F32) return go(swiglu_tag, Eight{}, Two{}, Four{}, One{});
        }
    };
    if (g.swiglu) pick(std::true_type{});
    else pick(std::false_type{});
    return refused ? hipErrorInvalidValue : hipGetLastError();
}

hipError_t launch_grouped_f32(const GroupedArgs& g, WeightKind wk, hipStream_t s) {
    switch (wk) {
        case WeightKind::F32: return launch_f32_t<float>(g, s);
        case WeightKind::BF16: return launch_f32_t<bf16_t>(g, s);
        case WeightKind::I8: return launch_f32_t<int8_t>(g, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace rbmoe
