// Launch interfaces between the C ABI (rbmoe_api.hip) and the kernel files.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <atomic>
#include <stddef.h>
#include <stdint.h>

#include "rbmoe_device.h"

namespace rbmoe {

// A kernel attribute is set once per device.  `done` has one bit per device; setting an attribute twice is
// harmless, so two threads that race here only repeat the call.  Devices past the 64th set it on every launch.
template <typename F>
inline hipError_t once_per_device(std::atomic<unsigned long long>& done, F&& set) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0ull;
    if (bit && (done.load(std::memory_order_acquire) & bit)) return hipSuccess;
    e = set();
    if (e == hipSuccess && bit) done.fetch_or(bit, std::memory_order_release);
    return e;
}


// Kernel durations the way a kernel trace reports them: while a KernelTimer is installed on the calling thread,
// every forward-path launch below carries its own start and stop events (hipExtLaunchKernelGGL), which receive the
// begin and end time stamps of that dispatch itself - no launch gap, no event-pair overhead.  Up to kMaxTimedLaunches
// launches per timer; further ones are plain launches.
constexpr int kMaxTimedLaunches = 4;
struct KernelTimer {
    hipEvent_t ev[2 * kMaxTimedLaunches] = {};
    int used = 0;
};
extern thread_local KernelTimer* g_kernel_timer;  // null (the default): plain launches
#define RB_LAUNCH(kernel, grid, block, lds, stream, ...)                                                        \
    do {                                                                                                        \
        ::rbmoe::KernelTimer* const kt_ = ::rbmoe::g_kernel_timer;                                              \
        if (kt_ != nullptr && kt_->used < ::rbmoe::kMaxTimedLaunches) {                                         \
            hipExtLaunchKernelGGL(kernel, grid, block, lds, stream, kt_->ev[2 * kt_->used],                     \
                                  kt_->ev[2 * kt_->used + 1], 0, __VA_ARGS__);                                  \
            ++kt_->used;                                                                                        \
        } else {                                                                                                \
            hipLaunchKernelGGL(kernel, grid, block, lds, stream, __VA_ARGS__);                                  \
        }                                                                                                       \
    } while (0)

// Tokens owned by one router / dispatch block: a block owns a contiguous slot range (slots are numbered
// token * k + rank).  The kernels that take a whole batch's rows at once use 8, 16 or 32 tokens a block, by what fills
// the chip (plan_router); the others 32.
constexpr int kRouterTokens = 32;
constexpr int kMinRouterTokens = 8;
constexpr int kRouterThreads = 512;     // router_kernel workgroup
constexpr int kRouterWaves = kRouterThreads / 64;

// Largest expert count and top-k the routing kernels are laid out for.
constexpr int kMaxExperts = 256;
constexpr int kMaxTopK = 32;

size_t router_lds_bytes(int E, int k);
constexpr int kMaxRouterLds = 160 * 1024;  // LDS per workgroup on gfx950

struct RouterArgs {
    const void* x;       // [T, d] f32 or bf16
    const float* wr;     // [E, d] f32
    const float* bias;   // [E] or null
    const uint8_t* valid;  // [T] or null
    int T, d, E, k;
    float* P;            // [T, E]
    float* lse;          // [T]
    int* expert_of;      // [T*k]
    float* gate_of;      // [T*k]
    int* rank_in_block;  // [T*k]
    int* blockcnt;       // [nb, E]
    float* partial;      // [nb, E+1]
    void* rows16 = nullptr;  // f32 rows only: [T, d] bf16 copy of x written on the way (d a multiple of 8), or null
    bool allow_fused = true; // logits and everything behind them in one launch where the shapes allow
    int min_tokens = kMinRouterTokens;  // of a router block: the block tables are sized for these
    // a quantized router (Quantized::matmul_rhs_transposed, src/quantized.rs:55-62): int8 rows and one scale per row;
    // `wr` is then not read and the logits are (sum_c x[c] * f32(q[c]), in the reference's 32 lanes) * scale
    const int8_t* wq = nullptr;      // [E, d]
    const float* wscale = nullptr;   // [E]
    // Whether every router weight - of a quantized router: its whole number - is zero or a bf16 value of a magnitude from 2^-40 to
    // below 2^20.  Times a bf16 element from 2^-72 to below 2^80 it is then exact in f32, and no sum of such products overflows
    // or falls below 2^-126 on the way: the logits of bf16 rows may be taken by fused multiply-adds.  What the host knew when it chose
    // the launch, and no more: a launch recorded into a graph or kept for a replay runs again when other weights lie in `wr`.
    bool exact = false;
    // The same of the weights that lie there when the launch runs, beside them on the device (null: always true, as of whole numbers).
    const int* exact_now = nullptr;
    // The norm in front of the layer (RmsNorm::forward, src/norm.rs:41-61), for calls whose plan says `takes_norm`: `x`
    // holds the raw rows, the routing is decided on the normed ones, which are written to `xn_out` [T, d].
    const float* norm_w = nullptr;
    float norm_eps = 0.0f;
    void* xn_out = nullptr;
    // Arrival counters, all zero between launches (kDecodeCombineCounterStride apart, one a block of tokens), or null: where
    // a few tokens have many experts, several workgroups then share a block's experts out.
    int* arrive = nullptr;
};
// How a call is routed: tokens of a router block (what launch_dispatch needs to know), whether the launch applies the
// norm that `a` asks for, and whether it writes the bf16 copy of f32 rows for a quantized router too.  Made once per call,
// from the pointers that the launch will get: which kernel takes a call depends on their alignment, and the kernels'
// blocks differ in tokens.
struct RouterPlan {
    int block_tokens = 0;
    bool takes_norm = false;
    bool q8_writes_rows16 = false;
    // route_rows_kernel: experts whose router rows lie in LDS together (0: another kernel), LDS bytes
    int row_experts = 0;
    size_t row_lds = 0;
    bool row_exact = false;  // ... route_exact_kernel in its place
    int row_slice = 0;  // ... and experts of a workgroup, where a block's experts are shared out (0: they are not)
    bool operator==(const RouterPlan& o) const {
        return block_tokens == o.block_tokens && takes_norm == o.takes_norm && q8_writes_rows16 == o.q8_writes_rows16 &&
               row_experts == o.row_experts && row_lds == o.row_lds && row_slice == o.row_slice && row_exact == o.row_exact;
    }
};
RouterPlan plan_router(const RouterArgs& a, bool bf16);
// The plan of a call behind a norm (a.x: the raw rows): where no launch takes the norm along, `a` is turned to the normed
// rows, which the caller then makes first (`norm_apart`), and the plan is theirs.
RouterPlan plan_router_behind_norm(RouterArgs& a, const void* normed, bool bf16, bool* norm_apart);
bool router_takes(const RouterArgs& a, const RouterPlan& p, bool bf16);  // whether `p` is the plan of these arguments
hipError_t launch_router(const RouterArgs& a, const RouterPlan& p, bool bf16, hipStream_t s);  // refuses any other plan

struct DispatchArgs {
    const void* x;
    const int* expert_of;
    const int* rank_in_block;
    const int* blockcnt;   // [nb, E]    per-block histogram from the router kernel
    const float* partial;  // [nb, E+1]  per-block sums of probabilities and of lse^2
    int T, d, E, k;
    int block_tokens;      // tokens of a router block (RouterPlan)
    float w_aux, w_z;
    int tile_m;            // rows per tile of the grouped products
    int* counts;           // [E]
    int* offsets;          // [E+1]
    int* tile_expert;      // [max_tiles]
    int* tile_row0;
    int* tile_rows;
    int* ntiles;           // [1]
    float* losses;         // [2]
    int* blockbase;        // [nb, E]  scratch: slots of expert e routed by the blocks before block b; then E + 1 sums
    int* perm_slot;
    int* perm_token;
    int* inv_pos;
    void* xg;  // [T*k, d] or null (rows are then gathered by the consumer)
};
hipError_t launch_dispatch(const DispatchArgs& a, bool bf16, hipStream_t s);

// What the router leaves behind and the tables that follow from it (layout_device.h)
struct LayoutArgs {
    const int* blockcnt;
    const float* partial;
    int T, E, k, TB;
    float w_aux, w_z;
    int tile_m;
    int* counts;
    int* offsets;
    int* tile_expert;
    int* tile_row0;
    int* tile_rows;
    int* ntiles;
    float* losses;
};
// ... and the slots, for a gate/up launch that works out its own tiles and writes the tables on the way
struct RoutedSlots {
    const int* expert_of = nullptr;  // null: a dispatch launch has made the tables
    const int* rank_in_block = nullptr;
    int* perm_slot = nullptr;
    int* perm_token = nullptr;
    int* inv_pos = nullptr;
    uint32_t k_recip = 0;  // 2^32 / k rounded up (k > 1)
    int tb_shift = 0, tile_shift = 0;  // log2 of a router block's tokens, of a tile's rows
    LayoutArgs layout{};
};
// Whether the gate/up product can do the dispatch's work for these arguments, and what it then takes
bool dispatch_in_product_ok(const DispatchArgs& a);
RoutedSlots routed_slots(const DispatchArgs& a);

struct CombineArgs {
    const void* y;        // [R, d] expert output rows, activation dtype
    const void* yshared;  // [T, d] or null
    const void* residual; // [T, d] or null
    const int* inv_pos;   // [T*k]
    const float* gate_of; // [T*k]
    int T, d, k;
    void* out;            // [T, d]
    // y (and, with shared_in_parts, yshared) lies in so many parts (1, 2 or 4) in f32, part_rows (T) rows apart: a row is the sum of its
    // parts in order, rounded to the type that the rows have otherwise
    int parts = 1;
    bool shared_in_parts = false;
    int part_rows = 0;
    bool rows_bf16 = false;  // under f32 activations: y and yshared are bf16 (matrix-core products of a bf16 / int8 layer)
};
hipError_t launch_combine(const CombineArgs& a, bool bf16, hipStream_t s);

// RmsNorm::forward (src/norm.rs:41-61) over rows: out = (x * inverse_rms(row)) * weight, the sum of squares in
// index order
hipError_t launch_rmsnorm(const void* x, const float* weight, float eps, int T, int d, void* out, bool bf16,
                          hipStream_t s);

// ---------------------------------------------------------------------------
// Grouped expert products.  Rows of `a` are grouped by expert through the tile
// table written by the scan kernel; a tile never spans two experts.
//   out[row, n] = sum_c a[row, c] * w[expert][n, c]        (SWIGLU = false)
//   out[row, n] = silu(a . wg[n]) * (a . wu[n])            (SWIGLU = true; the
//       expert's weight block holds the F gate rows, then the F up rows)
// int8 weights carry one f32 scale per weight row; the product is
// (sum_c a*q) * scale as in the reference (src/quantized.rs:55-62).
// ---------------------------------------------------------------------------
enum class WeightKind : int { F32 = 0, BF16 = 1, I8 = 2 };

struct GroupedArgs {
    const void* a;          // [rows, K] activation dtype
    const int* row_index;   // null: row r of a tile is a[row0 + r]; else a[row_index[row0 + r]]
    const void* w;          // expert 0's weight block
    size_t w_expert_stride; // elements between experts
    const float* scales;    // int8: expert 0's scales, one per weight row
    size_t s_expert_stride;
    int N;                  // output columns (F for SWIGLU, d for the down product)
    int K;
    const int* tile_expert;
    const int* tile_row0;
    const int* tile_rows;
    const int* ntiles;
    int max_tiles;
    int routed_rows = 0, groups = 0;  // f32 rows: rows in all and groups of the tile table, for the choice of a tile
    int likely_tiles = 0;   // what *ntiles will be about, for the choice of a kernel (0: max_tiles)
    int dense_rows;         // >= 0: one group of this many rows, no tile table (shared expert)
    void* out;              // [rows, N] activation dtype
    void* gu_out = nullptr; // gate/up launches: [rows, 2N] pre-activations (gate | up) kept for a backward pass
    // down-shaped launches: [rows, 2N] pre-activations of the forward pass.  The product rows are
    // then taken as the gradient of the hidden rows and SwiGLU's backward is applied on the way out: the
    // gradients of the pre-activations go to `gu_out` [rows, 2N] and `out` is not written.
    const void* swiglu_grad_gu = nullptr;
    bool swiglu;
    // matrix-core launches: a second, dense group in the same launch (the shared expert); rows 0: none.  Its weights
    // are of the same kind; pre-activations are kept (`gu_out`) for both groups or for neither.
    struct Dense {
        const void* a = nullptr;  // [rows, K]
        const void* w = nullptr;
        const float* scales = nullptr;
        int N = 0, K = 0, rows = 0;
        void* out = nullptr;      // [rows, N]
        void* gu_out = nullptr;   // [rows, 2N]
    } dense2;
    int group_m;            // MFMA path: M-tiles per scheduling group (0 = default)
    int tile_m = 0;         // rows per tile of the tile table
    RoutedSlots slots;      // gate/up launches of the matrix-core kernels: in the place of tile table and row index
    // plain launches: the reduction shared out over so many workgroups a tile.  Part p of a row of `out` lies p * part_rows rows on (of
    // dense2.out p * dense2.rows), in f32 whatever the rows' type, and the row is the parts' sum in order.
    int parts = 1;
    int part_rows = 0;
};
hipError_t launch_grouped_generic(const GroupedArgs& a, bool act_bf16, WeightKind wk, int tile_m,
                                  hipStream_t s);
constexpr int kGenericTileM = 16;

// bf16 matrix-core path (bf16 activations; bf16 or int8 weights): weights repacked into
// matrix-core operand order (pack_weight_*) and streamed global -> registers, activations
// global -> LDS by DMA.  `w` must have been packed matrix by matrix.
constexpr int kStreamTileM = 128;
int stream_tile_m(int rows, int groups, int F, int d);  // rows of the tile table's tiles for so many routed rows: 128 or 160
bool stream_shape_ok(int N, int K);
int stream_parts(const GroupedArgs& a);  // GroupedArgs::parts for a plain launch where there is room for them
hipError_t launch_grouped_stream(const GroupedArgs& a, WeightKind wk, hipStream_t s);
void pack_weight_bf16(const uint16_t* src, int rows, int cols, uint16_t* dst);
void pack_weight_i8(const int8_t* src, int rows, int cols, int8_t* dst);

// Products over f32 rows at f32 accuracy on the bf16 matrix cores: plain row-major weights of any kind, any shape.
int f32_tile_m(int rows, int groups);  // rows of the tile table's tiles for so many routed rows: 32 or 64
bool f32_shape_ok(int N, int K);
int f32_workgroups(const GroupedArgs& a, WeightKind wk);  // about as many as the launch has
int f32_parts(const GroupedArgs& a, WeightKind wk);  // GroupedArgs::parts for a plain launch where there is room for them
bool f32_joins(int F, int Fs);  // whether a shared expert of width Fs may go into the launches of experts of width F
hipError_t launch_grouped_f32(const GroupedArgs& a, WeightKind wk, hipStream_t s);

// ---- backward pass: the kernels around the matrix products (backward_kernels.hip) --------
// dy[pos] = gate * gout[token(pos)], grad_gates[slot] = gout[token] . y[pos]; row widths: multiples of 16 bytes
hipError_t launch_scale_rows(const void* gout, const void* y, const int* perm_slot, const int* perm_token,
                             const float* gate_of, const int* offsets, int E, int d, int max_rows, void* dy,
                             float* grad_gates, bool bf16, hipStream_t s);
// out[e][M][N] += A_e^T . B_e over the rows of group e (counts/offsets), or over dense_rows rows when >= 0
hipError_t launch_grouped_tn(const void* a, int M, const void* b, const int* b_row_index, int N, const int* counts,
                             const int* offsets, int groups, int dense_rows, float* out, size_t out_expert_stride,
                             bool bf16, hipStream_t s);

// Weight gradients on the matrix cores (bf16 or f32 operands): out[e] += A_e^T . B_e with the rows of a group cut into
// chunks.  How an expert far above the average share is handled:
//   None     one chunk per expert (a skewed load then serialises the launch)
//   Ordered  cut into several chunks; the first adds in place, the others store partial matrices (`partial`) that
//            a second kernel adds in chunk order: identical bits run to run
//   Atomic   cut into several chunks that all add with f32 atomics, in whatever order they arrive
// `overwrite`: out is known to hold zeros, whatever its bytes are, and is written instead of added to.
// `chunks` is scratch of weight_grad_table_ints(...) ints, `partial` of weight_grad_partial_bytes(...) bytes
// (a smaller buffer is legal: the launch then cuts less).
enum class WgradSplit : int { None = 0, Ordered = 1, Atomic = 2 };
bool weight_grad_shape_ok(int M, int N, bool bf16);
int weight_grad_max_chunks(int groups, int total_rows);
int weight_grad_table_ints(int groups, int total_rows);
size_t weight_grad_partial_bytes(int M, int N, int groups, int dense_rows, int total_rows, bool bf16);
// ... for a buffer that serves every launch of 1 .. max_tokens tokens (rows_per_token rows each; dense: rows = tokens)
size_t weight_grad_partial_bytes_upto(int M, int N, int groups, bool dense, int max_tokens, int rows_per_token,
                                      bool bf16);
// `part`: the chunk table is a launch of its own in front of the product and depends on nothing but counts and
// offsets - a caller may have it computed early, on another stream (TableOnly), and later issue the product with
// the same arguments (ProductOnly) once that launch has completed.
enum class WgradPart : int { Both = 0, TableOnly = 1, ProductOnly = 2 };
hipError_t launch_weight_grad(const void* a, int M, const void* b, int N, const int* counts, const int* offsets,
                              int groups, int dense_rows, int total_rows, WgradSplit split_mode, bool overwrite,
                              int* chunks, float* partial, size_t partial_bytes, float* out, size_t out_expert_stride,
                              bool bf16, hipStream_t s, WgradPart part = WgradPart::Both);

// gates -> probabilities -> logits, with the gradients of the two auxiliary losses
hipError_t launch_route_backward(const float* P, const float* lse, const int* expert_of, const float* grad_gates,
                                 const int* counts, const int* offsets, int T, int E, int k, float w_aux, float w_z,
                                 float* dlogits, hipStream_t s);
// grad_router += dlogits^T . x (through `partial`, router_grad_chunks(max_tokens) * E * d floats) and
// dxr = dlogits . wr
int router_grad_chunks(int max_tokens);
int router_grad_max_tokens();  // launch_router_grad refuses more rows than this
hipError_t launch_router_grad(const float* dlogits, const void* x, const float* wr, int T, int d, int E,
                              float* partial, float* grad_router, void* dxr, bool bf16, hipStream_t s);
// RmsNorm::backward (src/norm.rs:63-121): grad_input = d(norm)/dx applied to `up` (+ residual_grad when given),
// grad_weight += scale gradient (through `partial`, rmsnorm_grad_tiles(max_tokens) * d floats); `inv_rms` [T] scratch
int rmsnorm_grad_tiles(int max_tokens);
hipError_t launch_rmsnorm_backward(const void* x, const void* up, const float* weight, float eps,
                                   const void* residual_grad, int T, int d, void* grad_input, float* inv_rms,
                                   float* partial, float* grad_weight, bool bf16, hipStream_t s);
// out[i] = bf16(in[i]), nearest even; n a multiple of 8
hipError_t launch_cast_rows_bf16(const float* in, void* out, long long n, hipStream_t s);
hipError_t launch_fill_f32(float* p, float v, long long n, hipStream_t s);

// ---- decode-shaped path (a few tokens) -------------------------------------------
constexpr int kSmallRouteMaxTokens = 32;
constexpr int kSmallRouteMaxPairs = 2048;  // T * E
constexpr int kDecodeTileM = 32;

struct SmallRouteArgs {
    const void* x;
    const float* wr;
    const float* bias;
    const uint8_t* valid;
    int T, d, E, k;
    float w_aux, w_z;
    int tile_m;
    float* P;
    float* lse;
    int* expert_of;
    float* gate_of;
    int* counts;
    int* offsets;
    int* tile_expert;
    int* tile_row0;
    int* tile_rows;
    int* ntiles;
    float* losses;
    int* perm_slot;
    int* perm_token;
    int* inv_pos;
    // Optional norm in front of the layer (RmsNorm::forward, src/norm.rs:41-61): `x` holds the raw rows, the
    // kernel normalises them in LDS, routes on the normed rows and writes them to `xn_out` [T, d].  Only for
    // calls whose rows are staged in LDS (small_route_stages_rows).
    const float* norm_w = nullptr;
    float norm_eps = 0.0f;
    void* xn_out = nullptr;
    // f32 rows only: a bf16 copy [T, d] of the rows the routing is decided on (after the norm, if any), for the
    // matrix-core products; only for calls whose rows are staged in LDS (small_route_stages_rows)
    void* rows16 = nullptr;
};
bool small_route_stages_rows(const void* x, const float* wr, int T, int d, int E, bool bf16);
bool small_route_ok(int T, int E, int k);
hipError_t launch_route_small(const SmallRouteArgs& a, bool bf16, hipStream_t s);

// One launch covers the routed tiles (<= 32 rows each) and, when a_shared is set, the shared
// expert over rows [0, T_shared).  Weights are in the packed layout of pack_weight_*.
struct DecodeGemmArgs {
    const void* a;
    const int* row_index;
    const void* w;
    size_t w_expert_stride;  // elements
    const float* scales;
    size_t s_expert_stride;
    int N, K;
    const int* tile_expert;
    const int* tile_row0;
    const int* tile_rows;
    const int* ntiles;
    int max_tiles;
    void* out;
    int a_expert_rows = 0;  // rows of `a` per expert: a routed row r of expert e is a[e * a_expert_rows + row]
    const void* a_shared;
    const void* w_shared;
    const float* scales_shared;
    int N_shared, K_shared, T_shared;
    void* out_shared;
    int swiglu;
    // Down-shaped launches only, all null / zero otherwise: the combine folded into the launch.  The last workgroup
    // of a feature block to finish (one counter per block of 32 output features: zero before the launch, zero
    // again after it) sums that block's columns for every token - the token's expert rows in ascending expert order,
    // a rounded multiply by the gate and a rounded add each, then the shared expert's row, then the residual - and
    // writes them to cmb_out.  Nobody waits for anybody: whoever arrives last does the work.
    int* cmb_counter = nullptr;           // block b's counter at [b * kDecodeCombineCounterStride]
    const int* cmb_inv_pos = nullptr;     // [T * k]
    const float* cmb_gate_of = nullptr;   // [T * k]
    const void* cmb_residual = nullptr;   // [T, N] bf16, or f32 when cmb_f32, or null
    void* cmb_out = nullptr;              // [T, N] bf16, or f32 when cmb_f32; null: no combine in this launch
    int cmb_T = 0, cmb_k = 0;
    int cmb_f32 = 0;
};
constexpr int kDecodeCombineMaxBlocks = 1024;  // feature blocks a folded combine has counters for
// ints between two blocks' counters: every block's arrivals go to a cache line - and an L2 channel - of their own
// (side by side in one line, the atomics of a launch's two hundred workgroups queue up behind one another)
constexpr int kDecodeCombineCounterStride = 64;
constexpr size_t kDecodeCombineCounterBytes = (size_t)kDecodeCombineMaxBlocks * kDecodeCombineCounterStride * 4;
// ... whose last word, in a cache line that no counter shares, is the layer's RouterArgs::exact_now
constexpr int kRouterExactWord = kDecodeCombineMaxBlocks * kDecodeCombineCounterStride - 1;
bool decode_shape_ok(int N, int K);
hipError_t launch_decode_gemm(const DecodeGemmArgs& g, WeightKind wk, hipStream_t s);
// Routing and gate/up products in one launch: every expert's gate/up product over all T rows, hidden rows to g.out as
// [E][T, N]; the shared expert as in launch_decode_gemm.  g.a / g.a_shared: the call's rows as they are (a.x), f32 or
// bf16, raw when the routing applies a norm - the products then take the normed rows on the way.  P, lse, expert_of and
// gate_of are written, nothing else of the routing (DecodeLayoutArgs).
bool decode_front_ok(const RouterArgs& a, bool bf16);
hipError_t launch_decode_front(const RouterArgs& a, const DecodeGemmArgs& g, bool bf16, WeightKind wk, hipStream_t s);
// The tables and losses of a call routed by launch_decode_front.
struct DecodeLayoutArgs {
    const float* P;
    const float* lse;
    const int* expert_of;
    const uint8_t* valid;
    int T, E, k;
    float w_aux, w_z;
    int *counts, *offsets, *tile_expert, *tile_row0, *tile_rows, *ntiles;
    float* losses;
    int *perm_slot, *perm_token, *inv_pos;
};
hipError_t launch_decode_layout(const DecodeLayoutArgs& a, hipStream_t s);
// The down product behind launch_decode_front with the combine folded in (g as for launch_decode_gemm: cmb_* set,
// a_expert_rows = tokens of the call; expert rows to g.out in SLOT order), one row of workgroups per EXPERT instead of per
// entry of the tile table: a workgroup knows its weights from its place in the grid and requests them at once, and learns
// its rows from t.expert_of behind them.  An expert without rows costs its weights' bytes.  The tables and losses of `t` are
// made beside the products.
bool decode_down_by_expert_ok(const DecodeGemmArgs& g, int E, int T, int k);
hipError_t launch_decode_down_by_expert(const DecodeGemmArgs& g, const DecodeLayoutArgs& t, WeightKind wk, hipStream_t s);
// The same for a call of a row or two, where a workgroup takes all of a column block's rows; also behind launch_route_small
// (a_expert_rows 0: hidden rows by position, expert rows too, and the tables are there already).
bool decode_down_few_ok(const DecodeGemmArgs& g, WeightKind wk, int T, int k);
hipError_t launch_decode_down_few(const DecodeGemmArgs& g, const DecodeLayoutArgs& t, WeightKind wk, hipStream_t s);

}  // namespace rbmoe
