// C ABI of the gfx950 mixture-of-experts layer (see include/rbmoe.h).
//
// Host-side orchestration only: configuration checks, weight upload and
// conversion, workspace, and the launch sequence of one forward pass
//   router -> scan -> dispatch -> gate/up (+SwiGLU) -> down -> shared -> combine
// which follows MoeLayer::forward_train (reference src/moe.rs:243-341) stage by
// stage without any host round trip between the stages.  There is no CPU
// fallback: without a usable GPU every device entry point fails.
#include "../../include/rbmoe.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "host_io.h"
#include "rbmoe_kernels.h"

using namespace rbmoe;

thread_local rbmoe::KernelTimer* rbmoe::g_kernel_timer = nullptr;

// Scratch of rbmoe_forward_static: device memory that exists without any allocation call.  Every GPU the library
// runs on holds its own copy of the array, at its own address, until the process ends.  In host code the
// array's name is only a handle for hipGetSymbolAddress: rbmoe_ctx_create resolves it once per device and host
// code uses the resolved pointer from then on.
// (No `used` attribute: the compiler makes a static device variable visible to the runtime's lookup by name
// because host code takes its address below, and only then; marked `used` it stays a local symbol, which
// hipGetSymbolAddress cannot find.)
static __device__ __align__(256) unsigned char rbmoe_static_scratch[RBMOE_STATIC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};  // per device: the address of rbmoe_static_scratch there

// With `device` current.  Resolved once per device and kept.
hipError_t static_scratch_of(int device, void** out) {
    *out = nullptr;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(rbmoe_static_scratch));
        if (e != hipSuccess) return e;
        g_scratch_ptr[device] = p;
    }
    *out = g_scratch_ptr[device];
    return hipSuccess;
}

thread_local std::string g_global_error;

size_t dtype_size(int dt) { return dt == RBMOE_F32 ? 4 : dt == RBMOE_BF16 ? 2 : 1; }

uint16_t host_f32_to_bf16(float f) {
    uint32_t b;
    std::memcpy(&b, &f, 4);
    if ((b & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((b >> 16) | 0x0040u);
    b += 0x7fffu + ((b >> 16) & 1u);
    return (uint16_t)(b >> 16);
}
// RouterArgs::exact: bf16 values, zeros or of magnitudes from 2^-40 to below 2^20.
bool router_weights_exact(const float* w, size_t n) {
    for (size_t i = 0; i < n; ++i) {
        uint32_t b;
        std::memcpy(&b, w + i, 4);
        const uint32_t exponent = (b >> 23) & 0xffu;
        if ((b & 0xffffu) != 0 || ((b & 0x7fffffffu) != 0 && (exponent < 127 - 40 || exponent >= 127 + 20))) return false;
    }
    return true;
}
float host_bf16_to_f32(uint16_t h) {
    uint32_t b = (uint32_t)h << 16;
    float f;
    std::memcpy(&f, &b, 4);
    return f;
}

std::string config_problem(const rbmoe_config* c) {
    char buf[256];
    // The first three are MoeConfig::validate (reference src/moe.rs:68-86), same wording.
    if (c->num_experts <= 0) return "a MoE layer needs at least one expert";
    if (c->experts_per_token <= 0 || c->experts_per_token > c->num_experts) {
        std::snprintf(buf, sizeof buf, "experts_per_token must be between 1 and num_experts (%d), got %d",
                      c->num_experts, c->experts_per_token);
        return buf;
    }
    if (c->d_ff <= 0) return "expert d_ff must be non-zero";
    if (c->d_model <= 0) return "d_model must be non-zero";
    if (c->shared_d_ff < 0) return "shared_d_ff must not be negative";
    if (c->weight_dtype != RBMOE_F32 && c->weight_dtype != RBMOE_BF16 && c->weight_dtype != RBMOE_I8)
        return "weight_dtype must be f32, bf16 or int8";
    if (c->act_dtype != RBMOE_F32 && c->act_dtype != RBMOE_BF16) return "act_dtype must be f32 or bf16";
    if (c->max_tokens < 0) return "max_tokens must not be negative";
    return "";
}

std::string limit_problem(const rbmoe_config* c) {
    char buf[256];
    if (c->num_experts > kMaxExperts) {
        std::snprintf(buf, sizeof buf, "more than %d experts (got %d)", kMaxExperts, c->num_experts);
        return buf;
    }
    if (c->experts_per_token > kMaxTopK) {
        std::snprintf(buf, sizeof buf, "experts_per_token above %d (got %d)", kMaxTopK, c->experts_per_token);
        return buf;
    }
    if ((int64_t)c->max_tokens * c->experts_per_token > (int64_t)1 << 28) return "max_tokens * experts_per_token above 2^28";
    return "";
}

}  // namespace

struct rbmoe_ctx {
    int device = 0;
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    // The backward pass runs the router's branch beside the weight gradients: a second stream (default
    // priority, like the first) forked from and joined to `stream` with two events.  Created on first use.
    hipStream_t side_stream = nullptr;
    hipEvent_t ev_fork = nullptr, ev_fork2 = nullptr, ev_join = nullptr, ev_tables = nullptr;
    // host calls: the routing of a forward is complete (recorded on `stream`), its tables are in host memory (recorded
    // on the side stream).  Created with the side stream.
    hipEvent_t ev_routed = nullptr, ev_fetched = nullptr;
    size_t budget_bytes = 0;
    size_t allocated = 0;
    void* static_scratch = nullptr;  // this device's copy of rbmoe_static_scratch (RBMOE_STATIC_SCRATCH_BYTES)
    std::string last_error;
    int refs = 1;  // the caller's handle + one per live layer; torn down when the last one goes
};

namespace {

struct Buf {
    void* p = nullptr;
    size_t bytes = 0;
};

int fail(rbmoe_ctx* ctx, int code, const std::string& msg) {
    if (ctx) ctx->last_error = msg;
    g_global_error = msg;
    return code;
}

int hip_fail(rbmoe_ctx* ctx, hipError_t e, const char* what) {
    std::string msg = std::string(what) + ": " + hipGetErrorString(e);
    if (e == hipErrorOutOfMemory) return fail(ctx, RBMOE_OUT_OF_MEMORY, msg);
    return fail(ctx, RBMOE_DEVICE_ERROR, msg);
}

#define HIP_TRY(ctx, expr)                                         \
    do {                                                           \
        hipError_t _e = (expr);                                    \
        if (_e != hipSuccess) return hip_fail((ctx), _e, #expr);   \
    } while (0)

}  // namespace

// Where one forward pass keeps its routing tables and expert rows: the layer's own workspace, or a carving of
// the static scratch array (rbmoe_forward_static).  The getters read the last forward's.
struct Work {
    float* P = nullptr;
    float* lse = nullptr;
    int* expert_of = nullptr;
    float* gate_of = nullptr;
    int* counts = nullptr;
    int* offsets = nullptr;
    int* tile_expert = nullptr;
    int* tile_row0 = nullptr;
    int* tile_rows = nullptr;
    int* ntiles = nullptr;
    float* losses = nullptr;
    int* perm_slot = nullptr;
    int* perm_token = nullptr;
    int* inv_pos = nullptr;
    void* h = nullptr;
    void* y = nullptr;
    void* hs = nullptr;
    void* ys = nullptr;
    void* hall = nullptr;  // hidden rows of every expert over every row, [E][T, F] (decode_front launches), or null
    void* x16 = nullptr;   // bf16 copy of f32 rows [T, d] (layers with cast_rows), or null
    int* cmb_counter = nullptr;  // arrival counters of a combine folded into the decode-shaped down launch (all zero between launches)
};

// Host memory of a call that is still under way: a pinned block, or plain memory when the pool is exhausted.
struct Staging {
    HostBlock block;
    std::unique_ptr<unsigned char[]> plain;
    unsigned char* p = nullptr;
    bool pinned() const { return block.p != nullptr; }
    bool take(size_t bytes) {
        block = HostBlock(bytes);
        plain.reset();
        if (!block.p) plain.reset(new (std::nothrow) unsigned char[bytes]);
        p = block.p ? static_cast<unsigned char*>(block.p) : plain.get();
        return p != nullptr;
    }
    void reset() {
        block.reset();
        plain.reset();
        p = nullptr;
    }
};

// The output of a host call between its begin and its finish.
struct PendingOut {
    bool any = false;
    hipStream_t stream = nullptr;
    Staging in, out;
    void* user = nullptr;      // where the rows go from out.p once the stream is done (null: they are written in place)
    size_t elements = 0;
    bool from_bf16 = false;    // out.p holds bf16 rows and the caller wants f32
    size_t element_bytes = 0;  // otherwise: a plain copy
};

struct rbmoe_layer {
    rbmoe_ctx* ctx = nullptr;
    PendingOut pending;
    hipEvent_t record_routed = nullptr;  // forward_impl records it once the routing tables are complete
    rbmoe_config cfg{};
    int Fs = 0;       // shared expert width
    // Expert widths as the kernels see them: the matrix-core kernels take whole tiles, so a width between two multiples
    // of the tile is rounded up and the extra gate and up rows and down columns are zero (their hidden values are
    // silu(0) * 0 = 0 and add nothing).  Equal to the true widths where nothing is rounded.
    int Fw = 0, Fsw = 0;
    // Laid out as small as the kernels allow, because the memory budget, the memory or a limit of the rounded widths would
    // refuse the layer otherwise: true widths, router blocks of one size, no room for the routing beside the products of
    // a layer with many experts.
    bool tight = false;
    int max_T = 0;
    int max_S = 0;
    int max_nb = 0;
    int max_tiles = 0;
    bool force_generic = false;
    bool explicit_gather = false;  // materialise the gathered rows instead of gathering in the product
    bool use_stream = false;   // bf16 matrix-core kernels (packed weights); otherwise the generic kernels
    // f32 rows on the boundary of a layer with bf16 / int8 weights: the router reads the f32 rows, the expert
    // products run on the bf16 matrix cores over a bf16 copy of the rows (nearest even) that the routing kernels
    // write on the way, hidden and expert rows are bf16, and the combine sums them into f32 again
    bool cast_rows = false;
    bool use_f32_mc = false;   // all-f32 layer of whole tiles: the kernel set "mfma_f32"
    bool f32_rows = false;     // products over f32 rows at f32 accuracy (launch_grouped_f32): with use_f32_mc, and without it
                               // (the kernel name is then "generic") whatever the weights and widths
    bool decode_path = true;   // few tokens: launches that stream every touched weight once
    bool decode_front = true;  // ... the routing beside the gate/up products where that pays (decode_front_pays)
    bool shared_beside = true; // large batches: the shared expert's products on the side stream, beside the routing
    bool fused_router = true;  // logits and everything behind them in one launch where the shapes allow
    bool decode_fold = true;   // decode-shaped calls: the combine inside the down launch
    bool decode_down_by_expert = true;  // behind a decode_front launch: the down launch's workgroup rows are experts, not tile-table entries
    bool last_front = false;   // the last forward's hidden rows are per expert over all rows (Work::hall)
    bool last_by_slot = false; // ... and its expert rows lie in slot order
    bool last_few = false;     // ... by launch_decode_down_few
    int last_parts = 1;          // ... the parts that the last forward's expert rows lie in (CombineArgs::parts)
    int group_m = 0;
    const char* kernel_name = "none";
    int last_T = -1;
    int last_tile_m = kGenericTileM;  // rows per tile of the last forward's tile table
    Work last;  // tables of the last forward

    // weights
    Buf router;            // f32 [E, d]
    Buf router_q, router_s; // a quantized router: int8 [E, d], f32 scales [E] (`router` then holds the int8 values as f32)
    bool router_exact = false;  // RouterArgs::exact of the router that is set (a copy for the device: kRouterExactWord)
    bool router_q8 = false; // the layer routes with the quantized product (src/quantized.rs:55-62)
    bool quantize_router = false;  // f32 router data is quantized at upload (TransformerLm::quantize reaches the router too)
    int quant_rule = 0;     // f32 -> int8 at upload: 0 the checkpoint writer's rule, 1 the in-memory rule
    Buf wgu, wd;           // [E, 2F, d], [E, d, F] weight dtype
    Buf sgu, sd;           // int8 scales [E, 2F], [E, d]
    Buf swgu, swd;         // shared [2Fs, d], [d, Fs]
    Buf ssgu, ssd;         // shared scales
    // workspace
    Buf P, lse, expert_of, gate_of, rank_in_block, blockcnt, partial, blockbase;
    Buf counts, offsets, tile_expert, tile_row0, tile_rows, ntiles, losses;
    Buf perm_slot, perm_token, inv_pos;
    Buf xg, h, y, hs, ys;
    Buf x16;               // [max_T, d] bf16 copy of f32 rows (cast_rows)
    Buf hall;              // [E][min(max_T, 32), F] hidden rows of decode_front launches
    Buf cmbcnt;            // [kDecodeCombineMaxBlocks] arrival counters of the folded decode combine, kRouterExactWord
    // feed-forward norm in front of the layer (allocated by rbmoe_set_feed_forward_norm)
    Buf xn, norm_w;  // [max_T, d] activation dtype, [d] f32
    float norm_eps = 0.0f;
    bool norm_set = false;
    // training through the block step (allocated once both the norm and training mode are there)
    Buf xraw, dxn, inv_rms, norm_partial, g_norm;  // [T, d] x2 activation dtype, [T], [T/32][d], [d] f32
    bool last_was_block = false;
    // training (allocated by rbmoe_layer_enable_training)
    bool training = false;
    bool weights_set = false;
    Buf xc;                               // copy of the last input [T, d]
    const void* x_saved = nullptr;        // the last input as the backward pass reads it: xc, or the normed rows
    Buf gu, gus;                          // pre-activations (gate | up): [S, 2F], shared [T, 2Fs]
    Buf dy, dgu, dxg;                     // [S, d], [S, 2F], [S, d]
    Buf g16;                              // [T, d] bf16 copy of an f32 upstream gradient (cast_rows)
    Buf dgus, dxs;                        // shared: [T, 2Fs], [T, d]
    Buf grad_gates, ones, dlogits, dxr, rpartial;
    Buf g_router, g_gu, g_down, g_sgu, g_sdown;   // f32 weight gradients, accumulated
    Buf wg_chunks;                        // chunk table of the weight-gradient products
    Buf wg_partial;                       // partial matrices of cut experts (ordered accumulation)
    bool wgrad_generic = false, side_branch = true;
    WgradSplit wgrad_split = WgradSplit::Ordered;
    // The expert gradients count as zero without having been cleared (set by rbmoe_zero_grads): the next
    // backward pass overwrites them.
    bool grads_clear = false;
    Buf wdT, wguT, swdT, swguT;           // transposed packed weights: [E][F, d], [E][d, 2F], [Fs, d], [d, 2Fs]
    Buf st_gout, st_gin;
    // staging for the host entry point
    Buf st_x, st_out, st_valid, st_bias, st_res;
    std::vector<Buf*> all;
    hipEvent_t ev[RBMOE_NUM_STAGES + 1] = {};
    bool have_events = false;
    KernelTimer ktimer[RBMOE_NUM_STAGES];  // rbmoe_forward_kernel_times: events carried by the stages' own dispatches
    bool have_ktimers = false;
    // the launches of the last forward, stage by stage, for rbmoe_replay_stage (empty: the stage had no launch)
    std::function<hipError_t(hipStream_t)> replay[RBMOE_NUM_STAGES];
};

namespace {

struct Plan {
    std::vector<std::pair<Buf*, size_t>> items;
    size_t total = 0;
    void add(Buf* b, size_t bytes) {
        bytes = (bytes + 255) & ~(size_t)255;
        if (bytes == 0) bytes = 256;
        items.push_back({b, bytes});
        total += bytes;
    }
};

// Which kernel sets the layer's shapes and dtypes allow (and `force_generic` and `tight` do not rule out).
void choose_kernel_sets(rbmoe_layer* L) {
    const rbmoe_config* cfg = &L->cfg;
    L->use_stream = L->use_f32_mc = L->cast_rows = L->f32_rows = false;
    // Expert widths are rounded up to whole tiles (the model width is the caller's row pitch and is not): 64 columns
    // for the packed bf16 / int8 kernels, 32 for the f32 ones.  bf16 rows at other widths take the any-shape kernels, a
    // thirtieth of the matrix-core rate, so rounding pays up to four times the work and beyond.  All-f32 products at other
    // widths (launch_grouped_f32) fetch both operands element by element, and twice the work is still ahead: us a forward, d 512,
    // 8 experts, rounded / as they are: 682 (704) 64 rows 30.7 / 41.9, 1024 58.0 / 80.6, 4096 158 / 194; 130 (160) 1024 rows 36.6 /
    // 44.3; 40 (64) 32.0 / 36.9; 33 (64) 64 rows 27.6 / 31.6, 4096 52.4 / 59.0.
    auto rounded = [L](int f, int unit, int most) {
        const int up = (f + unit - 1) / unit * unit;
        return up <= most * f && !L->tight ? up : f;
    };
    const int unit = cfg->weight_dtype == RBMOE_F32 ? 32 : 64, most = cfg->weight_dtype == RBMOE_F32 ? 2 : 4;
    L->Fw = rounded(cfg->d_ff, unit, most);
    L->Fsw = rounded(L->Fs, unit, most);
    // bf16 matrix cores: bf16 activations, bf16 or int8 weights, widths that fit the packed layout
    // (f32 rows with bf16 / int8 weights - what a caller with f32 matrices and a quantized or bf16 checkpoint has -
    // take the same kernels over a bf16 copy of the rows)
    const bool mc = !L->force_generic && cfg->weight_dtype != RBMOE_F32;
    L->use_stream = mc && stream_shape_ok(L->Fw, cfg->d_model) && stream_shape_ok(cfg->d_model, L->Fw) &&
                    (!cfg->shared_expert ||
                     (stream_shape_ok(L->Fsw, cfg->d_model) && stream_shape_ok(cfg->d_model, L->Fsw)));

    L->use_f32_mc = !L->force_generic && cfg->act_dtype == RBMOE_F32 && cfg->weight_dtype == RBMOE_F32 &&
                    f32_shape_ok(L->Fw, cfg->d_model) && f32_shape_ok(cfg->d_model, L->Fw) &&
                    (!cfg->shared_expert || (f32_shape_ok(L->Fsw, cfg->d_model) && f32_shape_ok(cfg->d_model, L->Fsw)));
    {
        // the streaming kernel addresses activation rows with 32-bit byte offsets
        const size_t widest = (size_t)std::max(std::max(cfg->d_model, L->Fw), L->Fsw);
        const size_t rows = (size_t)cfg->max_tokens * (size_t)std::max(1, cfg->experts_per_token);
        if (rows * widest * 2 >= ((size_t)1 << 32)) L->use_stream = false;
    }
    if (cfg->act_dtype == RBMOE_F32 && L->use_stream) {
        // the bf16 copy is written in 8-element pieces of 16-byte aligned rows.  Rounding a width would also round the
        // rows: the products that such a layer has otherwise (f32_rows) keep input, hidden and expert rows in f32 (1e-5
        // against 3e-3), and the caller asked for f32 rows.
        const bool whole = L->Fw == cfg->d_ff && (!cfg->shared_expert || L->Fsw == L->Fs);
        if (cfg->d_model % 8 == 0 && whole) L->cast_rows = true;
        else L->use_stream = false;
    }
    L->f32_rows = cfg->act_dtype == RBMOE_F32 && !L->use_stream && !L->force_generic;
    if (!L->use_stream && !L->use_f32_mc) {
        // f32 rows over other weights: whole slices, like the all-f32 products.  us a forward, as they are / rounded, bf16 weights: d 512, 8
        // experts of 1365 (1376), 3 rows 47.0 / 28.3, 300 66.8 / 46.5, 8000 347 / 267; d 1024, 8 of 910 (928) and a shared one, 30 rows 51.5 /
        // 38.7, 2000 157 / 128; d 256, 8 of 341 (352), 3 rows 27.2 / 24.0, 8000 87.6 / 72.8, of 227 (256), 1000 rows 34.3 / 30.3; int8 alike.
        // Twice the work on narrow experts is made good by the whole pieces (of 33 (64), d 64, 3 and 3000 rows 21.9 / 21.1, 26.6 / 25.9; of 17
        // (32), d 1024, 48.8 / 46.9), and so it is where the model width has no whole slices and gate/up fetches element by element all
        // the same: d 33, of 50 (64), 25.1 / 25.0, 31.7 / 29.8; d 72, of 33, 24.2 / 23.3, 28.2 / 27.1; d 250, of 341, 36.5 / 32.9, 191 / 181; d 1000,
        // of 227, 42.2 / 39.8, 518 / 503 (int8 1044 / 1033); 216 such shapes 0.99 to 1.55 times as fast.
        // A training step over host matrices, d 256, 16 of 341 and a shared one, 200 rows 1450 / 1443, 4000 3590 / 2200.
        // Not under a memory budget, which may be laid out for layers of their true widths: several layers, or a norm set behind
        // training mode, which nothing makes room for.
        const bool rounds = L->f32_rows && (!L->ctx || L->ctx->budget_bytes == 0);
        L->Fw = rounds ? rounded(cfg->d_ff, 32, 2) : cfg->d_ff;
        L->Fsw = rounds ? rounded(L->Fs, 32, 2) : L->Fs;
    }
    const int block = L->tight ? kRouterTokens : kMinRouterTokens;  // tokens of the smallest router block
    L->max_nb = (cfg->max_tokens + block - 1) / block;
}

// What stands against the backward pass of a layer with these widths ("": nothing).
const char* training_widths_problem(const rbmoe_layer* L) {
    const rbmoe_config& c = L->cfg;
    const size_t d = c.d_model, F = L->Fw, Fs = L->Fsw, T = L->max_T, S = L->max_S;
    if (L->use_stream && c.weight_dtype == RBMOE_BF16) {
        if (!stream_shape_ok((int)d, (int)(2 * F)) || (c.shared_expert && !stream_shape_ok((int)d, (int)(2 * Fs))))
            return "expert width not supported by the backward products";
        // 32-bit byte offsets into the widest operand of the backward products: [S, 2F] bf16
        if (std::max(S * 2 * F, T * 2 * Fs) * 2 >= ((size_t)1 << 32))
            return "max_tokens x expert width too large for the backward products";
    } else if (L->use_f32_mc &&
               (!f32_shape_ok((int)d, (int)(2 * F)) || (c.shared_expert && !f32_shape_ok((int)d, (int)(2 * Fs))))) {
        return "expert width not supported by the backward products";
    }
    return "";  // (any other layer - odd widths, mixed dtypes - takes any widths in both directions: f32 rows through
                // launch_grouped_f32, bf16 rows on the any-shape kernels)
}

// Bytes for the down product's rows in parts: of at most half a million elements in quarters (stream_parts), or of 256 tiles of 64 x 128
// (f32_parts), 8 MB both, and no more than the layer's largest call.  Room of their own, so that whether a call's reduction is shared
// out, and with it the last bits of its rows, does not depend on the tokens that the layer has room for; behind the expert rows, since an
// allocation more would make a layer 20 us later.  Not in the tight layout or under a memory budget, which may be laid out for layers
// without it: there no reduction is shared out.
size_t parts_room(const rbmoe_layer* L) {
    const rbmoe_config& c = L->cfg;
    const bool may = (L->use_stream && c.d_model % 8 == 0) || (L->f32_rows && c.d_model % 4 == 0);
    if (!may || c.experts_per_token > 8 || L->tight || (L->ctx && L->ctx->budget_bytes)) return 0;
    const size_t rows = (size_t)L->max_S + (c.shared_expert ? (size_t)L->max_T : 0);
    return std::min(rows * c.d_model * 16, (size_t)8 << 20);
}

// Where that room begins in L->y.
size_t parts_offset(const rbmoe_layer* L) {
    const size_t bytes = (size_t)L->max_S * L->cfg.d_model * dtype_size(L->cfg.act_dtype);
    return (bytes + 255) & ~(size_t)255;
}

Plan make_plan(rbmoe_layer* L) {
    const rbmoe_config& c = L->cfg;
    const size_t E = c.num_experts, d = c.d_model, F = L->Fw, k = c.experts_per_token;
    const size_t Fs = L->Fsw, T = L->max_T, S = L->max_S, nb = L->max_nb;
    const size_t ws = dtype_size(c.weight_dtype), as = dtype_size(c.act_dtype);
    Plan p;
    p.add(&L->router, E * d * 4);
    p.add(&L->router_q, E * d);
    p.add(&L->router_s, E * 4);
    p.add(&L->wgu, E * 2 * F * d * ws);
    p.add(&L->wd, E * d * F * ws);
    if (c.weight_dtype == RBMOE_I8) {
        p.add(&L->sgu, E * 2 * F * 4);
        p.add(&L->sd, E * d * 4);
    }
    if (c.shared_expert) {
        p.add(&L->swgu, 2 * Fs * d * ws);
        p.add(&L->swd, d * Fs * ws);
        if (c.weight_dtype == RBMOE_I8) {
            p.add(&L->ssgu, 2 * Fs * 4);
            p.add(&L->ssd, d * 4);
        }
        p.add(&L->hs, T * Fs * as);
        p.add(&L->ys, T * d * as);
    }
    p.add(&L->P, T * E * 4);
    p.add(&L->lse, T * 4);
    p.add(&L->expert_of, S * 4);
    p.add(&L->gate_of, S * 4);
    p.add(&L->rank_in_block, S * 4);
    p.add(&L->blockcnt, nb * E * 4);
    p.add(&L->partial, nb * (E + 1) * 4);
    p.add(&L->blockbase, (nb * E + E + 1) * 4);
    p.add(&L->counts, E * 4);
    p.add(&L->offsets, (E + 1) * 4);
    p.add(&L->tile_expert, (size_t)L->max_tiles * 4);
    p.add(&L->tile_row0, (size_t)L->max_tiles * 4);
    p.add(&L->tile_rows, (size_t)L->max_tiles * 4);
    p.add(&L->ntiles, 8);
    p.add(&L->losses, 8);
    p.add(&L->perm_slot, S * 4);
    p.add(&L->perm_token, S * 4);
    p.add(&L->inv_pos, S * 4);
    if (L->cast_rows) p.add(&L->x16, T * d * 2);
    if (L->use_stream && E <= (L->tight ? std::min<size_t>(64, 16 * k) : 64))  // decode_front launches
        p.add(&L->hall, E * std::min<size_t>(T, kSmallRouteMaxTokens) * F * 2);
    p.add(&L->cmbcnt, kDecodeCombineCounterBytes);
    p.add(&L->xg, S * d * as);
    p.add(&L->h, S * F * as);
    p.add(&L->y, parts_offset(L) + parts_room(L));
    p.add(&L->st_x, T * d * as);
    p.add(&L->st_out, T * d * as);
    p.add(&L->st_res, T * d * as);
    p.add(&L->st_valid, T);
    p.add(&L->st_bias, E * 4);
    return p;
}

void free_layer_buffers(rbmoe_layer* L) {
    for (Buf* b : L->all) {
        if (b->p) {
            (void)hipFree(b->p);
            if (L->ctx && L->ctx->allocated >= b->bytes) L->ctx->allocated -= b->bytes;
            b->p = nullptr;
            b->bytes = 0;
        }
    }
    L->all.clear();
}

// The buffers of a new layer, cleared.  A failure leaves none of them behind.
int allocate_layer(rbmoe_layer* L) {
    rbmoe_ctx* ctx = L->ctx;
    Plan plan = make_plan(L);
    // Refuse before allocating anything, as the reference's budget check does
    // (src/param.rs:172-189).
    if (ctx->budget_bytes && ctx->allocated + plan.total > ctx->budget_bytes) {
        char buf[200];
        std::snprintf(buf, sizeof buf, "memory budget exceeded: estimated %zu MiB exceeds budget %zu MiB",
                      (ctx->allocated + plan.total + (1 << 20) - 1) >> 20, ctx->budget_bytes >> 20);
        return fail(ctx, RBMOE_MEMORY_BUDGET, buf);
    }
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    for (auto& it : plan.items) {
        void* p = nullptr;
        hipError_t e = hipMalloc(&p, it.second);
        if (e != hipSuccess) {
            size_t free_b = 0, total_b = 0;
            (void)hipGetLastError();
            (void)hipMemGetInfo(&free_b, &total_b);
            char buf[200];
            std::snprintf(buf, sizeof buf, "out of memory: an allocation of %zu MiB failed with %zu MiB free",
                          it.second >> 20, free_b >> 20);
            free_layer_buffers(L);
            return fail(ctx, RBMOE_OUT_OF_MEMORY, buf);
        }
        it.first->p = p;
        it.first->bytes = it.second;
        ctx->allocated += it.second;
        L->all.push_back(it.first);
        e = hipMemsetAsync(p, 0, it.second, ctx->stream);
        if (e != hipSuccess) {
            free_layer_buffers(L);
            return hip_fail(ctx, e, "hipMemsetAsync");
        }
    }
    const hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
        free_layer_buffers(L);
        return hip_fail(ctx, e, "hipStreamSynchronize");
    }
    return RBMOE_OK;
}

// A layer whose weights have not been set gives back what it holds beyond the tight layout, so that something further
// fits.  Every buffer of that layout is at most as large as the one it replaces, and where the smaller one cannot be had
// the layer keeps the larger.  A forward that has run on the zero weights is forgotten.
void make_tight(rbmoe_layer* L) {
    rbmoe_ctx* ctx = L->ctx;
    const Plan roomy = make_plan(L);
    L->tight = true;
    choose_kernel_sets(L);
    const Plan plan = make_plan(L);
    (void)hipStreamSynchronize(ctx->stream);
    L->last_T = -1;
    for (auto& r : L->replay) r = nullptr;
    for (const auto& was : roomy.items) {
        Buf* const b = was.first;
        size_t bytes = 0;
        for (const auto& it : plan.items)
            if (it.first == b) bytes = it.second;
        if (bytes == b->bytes) continue;
        void* p = nullptr;
        if (bytes != 0) {
            if (hipMalloc(&p, bytes) != hipSuccess) {
                (void)hipGetLastError();
                continue;
            }
            (void)hipMemsetAsync(p, 0, bytes, ctx->stream);
        }
        (void)hipFree(b->p);
        ctx->allocated -= b->bytes;
        ctx->allocated += bytes;
        b->p = p;
        b->bytes = bytes;
        if (bytes == 0) L->all.erase(std::find(L->all.begin(), L->all.end(), b));
    }
    (void)hipStreamSynchronize(ctx->stream);
}

}  // namespace

extern "C" {

const char* rbmoe_version(void) { return "rbmoe 0.1 (gfx950)"; }

const char* rbmoe_last_global_error(void) { return g_global_error.c_str(); }

int rbmoe_config_init(rbmoe_config* cfg, int32_t d_model, int32_t num_experts, int32_t experts_per_token,
                      int32_t d_ff) {
    if (!cfg) return fail(nullptr, RBMOE_NULL_POINTER, "cfg is NULL");
    std::memset(cfg, 0, sizeof *cfg);
    cfg->d_model = d_model;
    cfg->num_experts = num_experts;
    cfg->experts_per_token = experts_per_token;
    cfg->d_ff = d_ff;
    cfg->shared_expert = 0;
    cfg->shared_d_ff = 0;
    cfg->aux_loss_weight = 0.01f;
    cfg->router_z_loss_weight = 1e-3f;
    cfg->weight_dtype = RBMOE_F32;
    cfg->act_dtype = RBMOE_F32;
    cfg->max_tokens = 0;
    return RBMOE_OK;
}

int rbmoe_validate(const rbmoe_config* cfg, char* msg, size_t msg_cap) {
    if (!cfg) return fail(nullptr, RBMOE_NULL_POINTER, "cfg is NULL");
    std::string problem = config_problem(cfg);
    int code = RBMOE_INVALID_CONFIG;
    if (problem.empty()) {
        problem = limit_problem(cfg);
        code = RBMOE_UNSUPPORTED;
    }
    if (msg && msg_cap > 0) {
        std::snprintf(msg, msg_cap, "%s", problem.c_str());
    }
    if (problem.empty()) return RBMOE_OK;
    return fail(nullptr, code, problem);
}

int rbmoe_parameter_counts(const rbmoe_config* cfg, uint64_t* total, uint64_t* active) {
    if (!cfg) return fail(nullptr, RBMOE_NULL_POINTER, "cfg is NULL");
    const uint64_t d = cfg->d_model, E = cfg->num_experts, k = cfg->experts_per_token, F = cfg->d_ff;
    const uint64_t Fs = cfg->shared_d_ff > 0 ? cfg->shared_d_ff : cfg->d_ff;
    const uint64_t expert = 3 * d * F;
    const uint64_t shared = cfg->shared_expert ? 3 * d * Fs : 0;
    const uint64_t router = E * d;
    if (total) *total = router + E * expert + shared;
    if (active) *active = router + k * expert + shared;
    return RBMOE_OK;
}

int rbmoe_ctx_create(int32_t device, size_t budget_mib, rbmoe_ctx** out) {
    if (!out) return fail(nullptr, RBMOE_NULL_POINTER, "out is NULL");
    *out = nullptr;
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0) {
        (void)hipGetLastError();
        return fail(nullptr, RBMOE_BACKEND_UNAVAILABLE,
                    std::string("no usable HIP device: ") + (e != hipSuccess ? hipGetErrorString(e) : "device count is 0"));
    }
    if (device < 0 || device >= n) return fail(nullptr, RBMOE_INVALID_CONFIG, "device index out of range");
    hipDeviceProp_t prop;
    HIP_TRY(nullptr, hipGetDeviceProperties(&prop, device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(nullptr, RBMOE_UNSUPPORTED, std::string("kernels are built for gfx950, device is ") + prop.gcnArchName);
    HIP_TRY(nullptr, hipSetDevice(device));
    void* scratch = nullptr;
    HIP_TRY(nullptr, static_scratch_of(device, &scratch));
    rbmoe_ctx* ctx = new rbmoe_ctx();
    ctx->device = device;
    ctx->static_scratch = scratch;
    ctx->budget_bytes = budget_mib << 20;
    hipError_t se = hipStreamCreateWithFlags(&ctx->own_stream, hipStreamNonBlocking);
    if (se != hipSuccess) {
        delete ctx;
        return hip_fail(nullptr, se, "hipStreamCreateWithFlags");
    }
    ctx->stream = ctx->own_stream;
    host_pool_hold();
    *out = ctx;
    return RBMOE_OK;
}

static void ctx_release(rbmoe_ctx* ctx) {
    if (!ctx || --ctx->refs > 0) return;
    if (ctx->side_stream) {
        (void)hipStreamSynchronize(ctx->side_stream);
        (void)hipStreamDestroy(ctx->side_stream);
    }
    if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
    if (ctx->ev_fork2) (void)hipEventDestroy(ctx->ev_fork2);
    if (ctx->ev_join) (void)hipEventDestroy(ctx->ev_join);
    if (ctx->ev_tables) (void)hipEventDestroy(ctx->ev_tables);
    if (ctx->ev_routed) (void)hipEventDestroy(ctx->ev_routed);
    if (ctx->ev_fetched) (void)hipEventDestroy(ctx->ev_fetched);
    if (ctx->own_stream) {
        (void)hipStreamSynchronize(ctx->own_stream);
        (void)hipStreamDestroy(ctx->own_stream);
    }
    delete ctx;
    host_pool_release();
}

// Layers keep their context alive: destroying the context while layers exist
// only drops the caller's reference.
void rbmoe_ctx_destroy(rbmoe_ctx* ctx) { ctx_release(ctx); }

int rbmoe_ctx_set_stream(rbmoe_ctx* ctx, void* hip_stream) {
    if (!ctx) return fail(nullptr, RBMOE_NULL_POINTER, "ctx is NULL");
    ctx->stream = hip_stream ? static_cast<hipStream_t>(hip_stream) : ctx->own_stream;
    return RBMOE_OK;
}

int rbmoe_synchronize(rbmoe_ctx* ctx) {
    if (!ctx) return fail(nullptr, RBMOE_NULL_POINTER, "ctx is NULL");
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return RBMOE_OK;
}

const char* rbmoe_last_error(const rbmoe_ctx* ctx) { return ctx ? ctx->last_error.c_str() : g_global_error.c_str(); }

int rbmoe_layer_create(rbmoe_ctx* ctx, const rbmoe_config* cfg, rbmoe_layer** out) {
    if (!ctx || !cfg || !out) return fail(ctx, RBMOE_NULL_POINTER, "ctx, cfg or out is NULL");
    *out = nullptr;
    std::string problem = config_problem(cfg);
    if (!problem.empty()) return fail(ctx, RBMOE_INVALID_CONFIG, problem);
    problem = limit_problem(cfg);
    if (!problem.empty()) return fail(ctx, RBMOE_UNSUPPORTED, problem);
    if (cfg->max_tokens <= 0) return fail(ctx, RBMOE_INVALID_CONFIG, "max_tokens must be positive");
    if (router_lds_bytes(cfg->num_experts, cfg->experts_per_token) > (size_t)kMaxRouterLds)
        return fail(ctx, RBMOE_UNSUPPORTED, "router tile does not fit in LDS for this expert count and top-k");

    rbmoe_layer* L = new rbmoe_layer();
    L->ctx = ctx;
    L->cfg = *cfg;
    L->Fs = cfg->shared_d_ff > 0 ? cfg->shared_d_ff : cfg->d_ff;
    L->cfg.shared_d_ff = L->Fs;
    L->max_T = cfg->max_tokens;
    L->max_S = cfg->max_tokens * cfg->experts_per_token;
    L->max_tiles = L->max_S / kGenericTileM + cfg->num_experts + 1;
    // (behaviour switches keep their defaults here: rbmoe_layer_set_option changes them)
    int rc = RBMOE_OK;
    for (const bool tight : {false, true}) {
        L->tight = tight;
        choose_kernel_sets(L);
        rc = allocate_layer(L);
        if (rc != RBMOE_MEMORY_BUDGET && rc != RBMOE_OUT_OF_MEMORY) break;
    }
    if (rc != RBMOE_OK) {
        delete L;
        return rc;
    }
    ++ctx->refs;
    *out = L;
    return RBMOE_OK;
}

void rbmoe_layer_destroy(rbmoe_layer* L) {
    if (!L) return;
    rbmoe_ctx* owner = L->ctx;
    if (L->ctx) (void)hipStreamSynchronize(L->ctx->stream);
    if (L->have_events)
        for (auto& ev : L->ev)
            if (ev) (void)hipEventDestroy(ev);
    if (L->have_ktimers)
        for (auto& kt : L->ktimer)
            for (auto& ev : kt.ev)
                if (ev) (void)hipEventDestroy(ev);
    free_layer_buffers(L);
    delete L;
    ctx_release(owner);
}

int rbmoe_set_weight(rbmoe_layer* L, int32_t which, int32_t expert, const void* data, int32_t dtype,
                     const float* scales, int32_t rows, int32_t cols) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (!data) return fail(ctx, RBMOE_NULL_POINTER, "data is NULL");
    const rbmoe_config& c = L->cfg;
    const int E = c.num_experts, d = c.d_model, F = c.d_ff, Fs = L->Fs;
    int want_rows = 0, want_cols = 0;
    char* dst = nullptr;        // destination of the matrix, in weight-dtype elements
    float* sdst = nullptr;      // destination of the scales
    size_t elem_off = 0, scale_off = 0;
    bool is_router = false;
    switch (which) {
        case RBMOE_W_ROUTER:
            want_rows = E; want_cols = d; is_router = true;
            dst = static_cast<char*>(L->router.p);
            break;
        case RBMOE_W_GATE:
        case RBMOE_W_UP:
            want_rows = F; want_cols = d;
            if (expert < 0 || expert >= E) return fail(ctx, RBMOE_INVALID_CONFIG, "expert index out of range");
            elem_off = ((size_t)expert * 2 + (which == RBMOE_W_UP ? 1 : 0)) * L->Fw * d;
            scale_off = ((size_t)expert * 2 + (which == RBMOE_W_UP ? 1 : 0)) * L->Fw;
            dst = static_cast<char*>(L->wgu.p);
            sdst = static_cast<float*>(L->sgu.p);
            break;
        case RBMOE_W_DOWN:
            want_rows = d; want_cols = F;
            if (expert < 0 || expert >= E) return fail(ctx, RBMOE_INVALID_CONFIG, "expert index out of range");
            elem_off = (size_t)expert * d * L->Fw;
            scale_off = (size_t)expert * d;
            dst = static_cast<char*>(L->wd.p);
            sdst = static_cast<float*>(L->sd.p);
            break;
        case RBMOE_W_SHARED_GATE:
        case RBMOE_W_SHARED_UP:
            if (!c.shared_expert) return fail(ctx, RBMOE_INVALID_CONFIG, "the layer has no shared expert");
            want_rows = Fs; want_cols = d;
            elem_off = (size_t)(which == RBMOE_W_SHARED_UP ? 1 : 0) * L->Fsw * d;
            scale_off = (size_t)(which == RBMOE_W_SHARED_UP ? 1 : 0) * L->Fsw;
            dst = static_cast<char*>(L->swgu.p);
            sdst = static_cast<float*>(L->ssgu.p);
            break;
        case RBMOE_W_SHARED_DOWN:
            if (!c.shared_expert) return fail(ctx, RBMOE_INVALID_CONFIG, "the layer has no shared expert");
            want_rows = d; want_cols = Fs;
            dst = static_cast<char*>(L->swd.p);
            sdst = static_cast<float*>(L->ssd.p);
            break;
        default:
            return fail(ctx, RBMOE_INVALID_CONFIG, "unknown weight id");
    }
    if (rows != want_rows || cols != want_cols) {
        char buf[160];
        std::snprintf(buf, sizeof buf, "weight shape [%d, %d] does not match expected [%d, %d]", rows, cols,
                      want_rows, want_cols);
        return fail(ctx, RBMOE_INVALID_INPUT, buf);
    }
    const size_t n_given = (size_t)rows * cols;
    // The router is f32 whatever the experts' dtype - unless it is given as int8 rows with scales, or the layer
    // was told to quantize it like every other Linear (TransformerLm::quantize, src/transformer.rs:899-910, reaches
    // it through MoeLayer::linears_mut, src/moe.rs:491-500): the layer then routes with the quantized product.
    const bool router_to_i8 = is_router && (dtype == RBMOE_I8 || (L->quantize_router && dtype == RBMOE_F32));
    const int target = is_router ? (router_to_i8 ? RBMOE_I8 : RBMOE_F32) : c.weight_dtype;
    if (router_to_i8 && L->training)
        return fail(ctx, RBMOE_UNSUPPORTED, "the backward pass is not defined for a quantized router");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));  // no forward may still read the old weights

    std::vector<unsigned char> staged;
    std::vector<float> staged_scales;
    const void* src = data;
    if (dtype == target) {
        if (target == RBMOE_I8) {
            if (!scales) return fail(ctx, RBMOE_NULL_POINTER, "int8 weights need scales");
        }
    } else if (dtype == RBMOE_F32 && target == RBMOE_BF16) {
        staged.resize(n_given * 2);
        const float* f = static_cast<const float*>(data);
        uint16_t* o = reinterpret_cast<uint16_t*>(staged.data());
        for (size_t i = 0; i < n_given; ++i) o[i] = host_f32_to_bf16(f[i]);
        src = staged.data();
    } else if (dtype == RBMOE_BF16 && target == RBMOE_F32) {
        staged.resize(n_given * 4);
        const uint16_t* h = static_cast<const uint16_t*>(data);
        float* o = reinterpret_cast<float*>(staged.data());
        for (size_t i = 0; i < n_given; ++i) o[i] = host_bf16_to_f32(h[i]);
        src = staged.data();
    } else if (dtype == RBMOE_F32 && target == RBMOE_I8) {
        // Per row: scale = absmax / 127, then
        //   rule 0, the checkpoint writer's (reference src/transformer.rs:512-519, :1839-1847):
        //           q = clamp(round(w / scale)), a zero row stays zero;
        //   rule 1, the in-memory one of Quantized::from_matrix (src/quantized.rs:29-51), which
        //           TransformerLm::quantize applies: q = clamp(round(w * (1 / scale))).
        // `round` is f32::round: halves away from zero.  The two differ where the reciprocal's rounding moves a
        // quotient across a half.
        staged.resize(n_given);
        staged_scales.resize(rows);
        const float* f = static_cast<const float*>(data);
        int8_t* q = reinterpret_cast<int8_t*>(staged.data());
        for (int r = 0; r < rows; ++r) {
            float absmax = 0.0f;
            for (int cc = 0; cc < cols; ++cc) absmax = std::fmax(absmax, std::fabs(f[(size_t)r * cols + cc]));
            const float scale = absmax / 127.0f;
            staged_scales[r] = scale;
            const float inverse = scale > 0.0f ? 1.0f / scale : 0.0f;
            for (int cc = 0; cc < cols; ++cc) {
                const float w = f[(size_t)r * cols + cc];
                float v = L->quant_rule == 1 ? std::round(w * inverse) : (scale == 0.0f ? 0.0f : std::round(w / scale));
                v = std::fmin(127.0f, std::fmax(-127.0f, v));
                q[(size_t)r * cols + cc] = (int8_t)v;
            }
        }
        src = staged.data();
        scales = staged_scales.data();
    } else {
        return fail(ctx, RBMOE_UNSUPPORTED, "this conversion between weight dtypes is not supported");
    }
    if (is_router) {
        if (router_to_i8) {
            HIP_TRY(ctx, hipMemcpy(L->router_q.p, src, n_given, hipMemcpyHostToDevice));
            HIP_TRY(ctx, hipMemcpy(L->router_s.p, scales, (size_t)rows * 4, hipMemcpyHostToDevice));
            // ... and widened, for the products of large calls (logits_kernel)
            const int8_t* const q = static_cast<const int8_t*>(src);
            const std::vector<float> wide(q, q + n_given);
            HIP_TRY(ctx, hipMemcpy(L->router.p, wide.data(), n_given * 4, hipMemcpyHostToDevice));
        } else {
            HIP_TRY(ctx, hipMemcpy(L->router.p, src, n_given * 4, hipMemcpyHostToDevice));
        }
        L->router_q8 = router_to_i8;
        L->router_exact = router_to_i8 || router_weights_exact(static_cast<const float*>(src), n_given);
        const int exact_now = L->router_exact;
        HIP_TRY(ctx, hipMemcpy((int*)L->cmbcnt.p + kRouterExactWord, &exact_now, 4, hipMemcpyHostToDevice));
        L->weights_set = true;
        return RBMOE_OK;
    }
    const size_t es = dtype_size(target);
    const int scale_rows = rows;  // (the scales of rows added below stay zero)
    std::vector<unsigned char> widened;
    {
        const bool shared_w = which >= RBMOE_W_SHARED_GATE;
        const bool is_down = which == RBMOE_W_DOWN || which == RBMOE_W_SHARED_DOWN;
        const int wide = shared_w ? L->Fsw : L->Fw;
        const int to_rows = is_down ? rows : wide, to_cols = is_down ? wide : cols;
        if (to_rows != rows || to_cols != cols) {  // the width the kernels see: zero rows below, zero columns behind
            widened.assign((size_t)to_rows * to_cols * es, 0);
            for (int r = 0; r < rows; ++r)
                std::memcpy(widened.data() + (size_t)r * to_cols * es,
                            static_cast<const unsigned char*>(src) + (size_t)r * cols * es, (size_t)cols * es);
            src = widened.data();
            rows = to_rows;
            cols = to_cols;
        }
    }
    const size_t n = (size_t)rows * cols;
    const void* const plain_src = src;  // row-major, in the weight dtype
    std::vector<unsigned char> packed;
    if (L->use_stream && !is_router) {
        // operand order of the matrix cores, matrix by matrix (same offsets, different inner layout)
        packed.resize(n * es);
        if (target == RBMOE_BF16)
            pack_weight_bf16(static_cast<const uint16_t*>(src), rows, cols, reinterpret_cast<uint16_t*>(packed.data()));
        else
            pack_weight_i8(static_cast<const int8_t*>(src), rows, cols, reinterpret_cast<int8_t*>(packed.data()));
        src = packed.data();
    }
    HIP_TRY(ctx, hipMemcpy(dst + elem_off * es, src, n * es, hipMemcpyHostToDevice));
    if (target == RBMOE_I8)
        HIP_TRY(ctx, hipMemcpy(sdst + scale_off, scales, (size_t)scale_rows * 4, hipMemcpyHostToDevice));
    L->weights_set = true;
    if (L->training && !is_router) {
        // The backward products multiply by the weight itself, not by its transpose (grad_input =
        // grad_output . W, src/param.rs:822-823): keep a transposed copy in the layout the product kernels
        // read.  Gate and up share one matrix [d, 2F] (gate^T in columns [0, F), up^T in [F, 2F)) so that
        // dX = dG . Wg + dU . Wu is one product.
        const bool shared_w = which >= RBMOE_W_SHARED_GATE;
        const bool is_down = which == RBMOE_W_DOWN || which == RBMOE_W_SHARED_DOWN;
        const bool is_up = which == RBMOE_W_UP || which == RBMOE_W_SHARED_UP;
        const int Fw = shared_w ? L->Fsw : L->Fw;
        if (target == RBMOE_F32) {
            // plain row-major f32, as the f32 product kernel reads its weights
            const float* f = static_cast<const float*>(src);
            std::vector<float> tr(n);
            for (int r = 0; r < rows; ++r)
                for (int cc = 0; cc < cols; ++cc) tr[(size_t)cc * rows + r] = f[(size_t)r * cols + cc];
            if (is_down) {
                float* tdst = static_cast<float*>(shared_w ? L->swdT.p : L->wdT.p) + (shared_w ? 0 : (size_t)expert * Fw * d);
                HIP_TRY(ctx, hipMemcpy(tdst, tr.data(), n * 4, hipMemcpyHostToDevice));
            } else {
                float* base = static_cast<float*>(shared_w ? L->swguT.p : L->wguT.p) +
                              (shared_w ? 0 : (size_t)expert * d * 2 * Fw) + (is_up ? Fw : 0);
                HIP_TRY(ctx, hipMemcpy2D(base, (size_t)2 * Fw * 4, tr.data(), (size_t)Fw * 4, (size_t)Fw * 4, (size_t)d,
                                         hipMemcpyHostToDevice));
            }
        } else if (!L->use_stream) {
            // plain row-major bf16, as the any-shape product kernel reads its weights
            const uint16_t* h = static_cast<const uint16_t*>(src);
            std::vector<uint16_t> tr(n);
            for (int r = 0; r < rows; ++r)
                for (int cc = 0; cc < cols; ++cc) tr[(size_t)cc * rows + r] = h[(size_t)r * cols + cc];
            if (is_down) {
                uint16_t* tdst = static_cast<uint16_t*>(shared_w ? L->swdT.p : L->wdT.p) + (shared_w ? 0 : (size_t)expert * Fw * d);
                HIP_TRY(ctx, hipMemcpy(tdst, tr.data(), n * 2, hipMemcpyHostToDevice));
            } else {
                uint16_t* base = static_cast<uint16_t*>(shared_w ? L->swguT.p : L->wguT.p) +
                                 (shared_w ? 0 : (size_t)expert * d * 2 * Fw) + (is_up ? Fw : 0);
                HIP_TRY(ctx, hipMemcpy2D(base, (size_t)2 * Fw * 2, tr.data(), (size_t)Fw * 2, (size_t)Fw * 2, (size_t)d,
                                         hipMemcpyHostToDevice));
            }
        } else {
            // packed bf16; column steps of 16 never straddle the two halves of [d, 2F]
            const uint16_t* const plain = static_cast<const uint16_t*>(plain_src);
            std::vector<uint16_t> tr(n), trp(n);
            for (int r = 0; r < rows; ++r)
                for (int cc = 0; cc < cols; ++cc) tr[(size_t)cc * rows + r] = plain[(size_t)r * cols + cc];
            pack_weight_bf16(tr.data(), cols, rows, trp.data());  // [cols, rows] matrix
            if (is_down) {
                char* tdst = static_cast<char*>(shared_w ? L->swdT.p : L->wdT.p) + (shared_w ? 0 : (size_t)expert * Fw * d * 2);
                HIP_TRY(ctx, hipMemcpy(tdst, trp.data(), n * 2, hipMemcpyHostToDevice));
            } else {
                // [d, Fw] packed as [d/32][Fw/16][512]; destination [d/32][2Fw/16][512]
                char* base = static_cast<char*>(shared_w ? L->swguT.p : L->wguT.p) +
                             (shared_w ? 0 : (size_t)expert * d * 2 * Fw * 2);
                const size_t half = (size_t)(Fw / 16) * 512;  // elements per row block and half
                for (int rb = 0; rb < d / 32; ++rb)
                    HIP_TRY(ctx, hipMemcpy(base + ((size_t)rb * 2 * half + (is_up ? half : 0)) * 2,
                                           trp.data() + (size_t)rb * half, half * 2, hipMemcpyHostToDevice));
            }
        }
    }
    return RBMOE_OK;
}

}  // extern "C"

namespace {

// The second stream of a context (default priority, like the first) and the events that fork it from and join it
// to the main one: the backward pass runs the router's branch there, the forward pass the shared expert.
int ensure_side_stream(rbmoe_ctx* ctx) {
    if (ctx->side_stream) return RBMOE_OK;
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    // all of them or none: a stream without its events would be used as if it were complete
    hipStream_t st = nullptr;
    hipEvent_t ev[6] = {};
    hipError_t e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
    for (int i = 0; i < 6 && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
    if (e != hipSuccess) {
        for (hipEvent_t x : ev)
            if (x) (void)hipEventDestroy(x);
        if (st) (void)hipStreamDestroy(st);
        return hip_fail(ctx, e, "creating the context's second stream");
    }
    ctx->side_stream = st;
    ctx->ev_fork = ev[0];
    ctx->ev_fork2 = ev[1];
    ctx->ev_join = ev[2];
    ctx->ev_tables = ev[3];
    ctx->ev_routed = ev[4];
    ctx->ev_fetched = ev[5];
    return RBMOE_OK;
}

// ints of one chunk table of a training layer's weight-gradient launches (the largest of them)
static size_t wgrad_table_ints(const rbmoe_layer* L) {
    const int E = L->cfg.num_experts;
    return (size_t)std::max(weight_grad_table_ints(E, L->max_S), weight_grad_table_ints(1, L->max_T));
}

Work work_of_layer(const rbmoe_layer* L) {
    Work w;
    w.P = (float*)L->P.p; w.lse = (float*)L->lse.p;
    w.expert_of = (int*)L->expert_of.p; w.gate_of = (float*)L->gate_of.p;
    w.counts = (int*)L->counts.p; w.offsets = (int*)L->offsets.p;
    w.tile_expert = (int*)L->tile_expert.p; w.tile_row0 = (int*)L->tile_row0.p; w.tile_rows = (int*)L->tile_rows.p;
    w.ntiles = (int*)L->ntiles.p; w.losses = (float*)L->losses.p;
    w.perm_slot = (int*)L->perm_slot.p; w.perm_token = (int*)L->perm_token.p; w.inv_pos = (int*)L->inv_pos.p;
    w.h = L->h.p; w.y = L->y.p; w.hs = L->hs.p; w.ys = L->ys.p;
    w.hall = L->hall.p;
    w.x16 = L->x16.p;
    w.cmb_counter = (int*)L->cmbcnt.p;
    return w;
}

// Whether a decode-shaped call of T tokens should take every expert's products without waiting for the routing: when most
// experts are about to be touched, or when the weights fetched for nothing cost less than the launch and the chain in
// front of the products that this saves.  us, routing in front / beside, at so many MB expected for nothing (top-2 of 8 to
// 32 experts):
//   bf16: d 512, 26 18.0 / 12.4; d 768, 29 18.3 / 15.2, 39 18.0 / 15.0, 47 26.3 / 25.7, 61 23.6 / 24.3, 80 19.6 / 22.8; d 512,
//     41 20.8 / 20.1, 46 19.9 / 20.0, 53 19.1 / 19.9; d 256, 41 24.5 / 25.0.
//   int8 (widened on the way, so a byte takes longer): d 512, 27 19.5 / 16.1, 30 19.0 / 15.8; d 768, 40 20.1 / 18.6; d 1024,
//     top-4, 22 25.8 / 25.7, 29 24.6 / 25.5, 39 23.8 / 25.3, 52 22.1 / 24.3.
//   where the routing alone would not hold its rows in LDS its chain grows with the tokens.  32 experts: d 768 of 704, 1
//     token, 97 23.7 / 25.6, 2, 91 24.8 / 25.4, 3, 86 31.2 / 25.5, 8, 62 37.0 / 27.6; d 1024, 2, 106 35.4 / 33.4, 3, 93 50.5 /
//     33.9; d 768 of 1408, 3, 189 31.0 / 40.0; 64 experts, d 1024, top-6, 8, 126 72.2 / 75.7.
//   with an RMSNorm in front, which every workgroup of the one launch does again before its products: d 256, 32 experts of
//     1408, 4 rows, 40 24.5 / 27.0, 8 rows, 41 28.0 / 30.8; d 512, 16 experts of 1408, 2 rows, 40 22.9 / 23.7, 4 rows, 41 24.4
//     / 26.6, 8 experts, 26 21.7 / 15.4; rows not held: 32 experts, d 1024, 3, 70 52.4 / 38.4, d 768, 3, 86 38.9 / 35.8; 64
//     experts, top-6, d 512, 4, 93 47.3 / 45.8, d 1024 with a shared expert, 8, 95 72.6 / 75.3, 7, 104 75.0 / 82.7.
bool decode_front_pays(const rbmoe_layer* L, int T, bool stages_rows, bool normed) {
    const rbmoe_config& c = L->cfg;
    const double E = c.num_experts, k = c.experts_per_token;
    if (T * k >= 2 * E) return true;
    const double untouched = E * std::pow(1.0 - k / E, T);
    const double cost = untouched * 3.0 * L->Fw * c.d_model * (c.weight_dtype == RBMOE_I8 ? 1.5 : 2.0);
    const double held = normed ? 38e6 : 42e6;  // what may be fetched for nothing where routing alone holds its rows
    return cost <= (stages_rows ? held : std::max(held, (normed ? 30e6 : 36e6) * std::min(T, 3)));
}

// Whether a few tokens' call is better off on the decode-shaped kernels than on the large-batch sequence, whose routing
// takes a workgroup per eight tokens and whose launches a few microseconds each.  us, decode against large-batch:
//   routing beside the products: its down launch sums slots one after the other.  Over 64 slots and 20 M weights a
//     matrix: d 1024, 16 experts of 1408, four a row, 17 rows 1.07 times as long as the large-batch launches, 32 rows 1.38;
//     32 experts of 1408, d 512, 1.11 / 1.42.  Fewer weights, later: 32 rows, four a row, 16 experts, d 768 (17 M) 50.8 / 43.0,
//     8 experts, d 1024 (12 M) 44.4 / 41.2.
//     Its routing workgroup takes every expert's row, the large-batch routing shares them out (plan_rows): from 32 K router
//     weights on and with 20 M weights a matrix, 32 experts of 704, d 1024, 4 to 32 rows 0.98 to 1.18, behind a norm 1.09 to
//     1.24; 64 experts of 704, d 512, 1.00 to 1.19, behind a norm 1.15 to 1.33, d 1024 with a shared expert 1.36 to 1.65; 24 K
//     (32 of 1408, d 768) 0.77 to 0.87, behind a norm 0.98 to 1.04.
//   routing alone in one workgroup, in front: its time grows with tokens x experts x width, steeply where the rows do not
//     fit its LDS.  d 1024, 16 experts of 1408: 1 row 0.68, 4 rows 0.83, 8 rows 0.97, behind a norm 0.84, 0.99, 1.08; 32 experts,
//     d 512, 4 rows 0.87 / 0.99, 6 rows 1.06 / 1.12; staged: 16 experts, d 768, 12 rows (147 K) 44.8 us / 43.3.  Over 32 experts
//     and 32 K router weights the routing that shares them out is ahead sooner: 64 experts, d 512, 1 row 0.89 / 0.99, 2 rows
//     1.05 / 1.19, 4 rows - / 1.56; d 1024, 1 row 1.38 / 1.54, 8 rows 3.2.
// Where the lines are known to be off: four experts a row and more than 72 slots (16 and 32 experts, 1.2 to 1.67; d 1024, 32 experts of 256,
// 32 rows 53.7 us / 32.1), a block step over 32 experts that are routed alone (d 768, 4 rows 43.6 / 29.4), int8, 8 experts, d 1024, 16 to 24
// rows (46.8 / 33.0), 32 experts of 704 at d 768 and of 1408 at d 256, 24 to 28 rows (1.1 to 1.26).
bool decode_front_beats_batch(const rbmoe_layer* L, int T) {
    const rbmoe_config& c = L->cfg;
    const int slots = T * c.experts_per_token, E = c.num_experts;
    const double weights = (double)E * L->Fw * c.d_model;
    return !((slots > 64 || E * c.d_model >= 32 * 1024) && weights > 20e6) && !(slots > 112 && weights > 11e6);
}
bool decode_alone_beats_batch(const rbmoe_layer* L, int T, bool stages_rows) {
    const long long E = L->cfg.num_experts, work = T * E * L->cfg.d_model;
    return work <= (E > 32 && E * L->cfg.d_model >= 32 * 1024 ? 40000 : stages_rows ? 160000 : 110000);
}

// The buffers of a decode-shaped forward of T tokens carved out of `base` (pieces of 256 bytes); returns the
// bytes used.  With base == nullptr only the size is computed.
size_t carve_decode_work(const rbmoe_layer* L, int T, bool front, unsigned char* base, Work* w) {
    const rbmoe_config& c = L->cfg;
    const size_t E = c.num_experts, d = c.d_model, F = L->Fw, k = c.experts_per_token, Fs = L->Fsw;
    const size_t S = (size_t)T * k, as = L->cast_rows ? 2 : dtype_size(c.act_dtype);
    const size_t tiles = S / kDecodeTileM + E + 1;
    size_t used = 0;
    auto take = [&](size_t bytes) -> void* {
        void* p = base ? base + used : nullptr;
        used += (std::max<size_t>(bytes, 1) + 255) & ~(size_t)255;
        return p;
    };
    Work v;
    // first, at the same place for every call and every layer: the arrival counters of the folded combine, which are
    // zero whenever no call is running (the array starts as zeros and every launch leaves them as it found them)
    v.cmb_counter = (int*)take(kDecodeCombineCounterBytes);
    v.P = (float*)take((size_t)T * E * 4); v.lse = (float*)take((size_t)T * 4);
    v.expert_of = (int*)take(S * 4); v.gate_of = (float*)take(S * 4);
    v.counts = (int*)take(E * 4); v.offsets = (int*)take((E + 1) * 4);
    v.tile_expert = (int*)take(tiles * 4); v.tile_row0 = (int*)take(tiles * 4); v.tile_rows = (int*)take(tiles * 4);
    v.ntiles = (int*)take(8); v.losses = (float*)take(8);
    v.perm_slot = (int*)take(S * 4); v.perm_token = (int*)take(S * 4); v.inv_pos = (int*)take(S * 4);
    v.h = take(S * F * as); v.y = take(S * d * as);
    if (front) v.hall = take(E * (size_t)T * F * 2);
    if (c.shared_expert) {
        v.hs = take((size_t)T * Fs * as);
        v.ys = take((size_t)T * d * as);
    }
    if (L->cast_rows) v.x16 = take((size_t)T * d * 2);
    if (w) *w = v;
    return used;
}

// The matrix-core products fetch their rows by LDS-DMA in 16-byte pieces (every row is a whole number of them).  A caller's
// rows that start off such a boundary are copied to the layer's own memory first.
bool starts_on_piece(const void* rows) { return reinterpret_cast<uintptr_t>(rows) % 16 == 0; }

// `norm_src` (block step): the raw rows; `x` is then the layer's buffer of normed rows, filled here - by the
// small-route kernel itself for a few tokens, by the norm kernel otherwise - before anything reads it.
// `static_scratch` (rbmoe_forward_static): this device's copy of the static scratch array; the call must then be
// decode-shaped, keeps every intermediate result there and touches none of the layer's workspace.
// What the tile table of so many routed rows will hold about: a last tile half full, or one tile each.
int likely_tiles(int rows, int E, int tile_m) { return std::max(rows / tile_m + E / 2, std::min(E, rows)); }

// `timing`: 0 none; 1 an event between the stages (rbmoe_forward_timed); 2 every stage's dispatches carry their own
// start and stop events (rbmoe_forward_kernel_times).
int forward_impl(rbmoe_layer* L, const void* x, int T, int cols, const uint8_t* valid, const float* router_bias,
                 const void* residual, void* out, int timing, const void* norm_src = nullptr,
                 void* static_scratch = nullptr) {
    const bool timed = timing != 0;
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    const rbmoe_config& c = L->cfg;
    const int E = c.num_experts, d = c.d_model, F = L->Fw, k = c.experts_per_token, Fs = L->Fsw;
    // MoeLayer::forward_train's width check (reference src/moe.rs:248-253)
    if (cols != d) {
        char buf[120];
        std::snprintf(buf, sizeof buf, "input length %d does not match expected length %d", cols, d);
        return fail(ctx, RBMOE_INVALID_INPUT, buf);
    }
    if (T < 0) return fail(ctx, RBMOE_INVALID_INPUT, "negative token count");
    if (T > L->max_T) {
        char buf[120];
        std::snprintf(buf, sizeof buf, "%d tokens exceed the layer's max_tokens %d", T, L->max_T);
        return fail(ctx, RBMOE_INVALID_INPUT, buf);
    }
    if (T > 0 && (!x || !out)) return fail(ctx, RBMOE_NULL_POINTER, "x or out is NULL");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    L->last_was_block = false;  // rbmoe_forward_block sets it once this call has succeeded
    const bool abf = c.act_dtype == RBMOE_BF16;
    const bool cast = L->cast_rows;  // f32 rows, bf16 matrix-core products over their bf16 copy
    const WeightKind wk = c.weight_dtype == RBMOE_F32 ? WeightKind::F32
                          : c.weight_dtype == RBMOE_BF16 ? WeightKind::BF16 : WeightKind::I8;
    if (timing == 1 && !L->have_events) {
        for (auto& ev : L->ev) HIP_TRY(ctx, hipEventCreate(&ev));
        L->have_events = true;
    }
    if (timing == 2 && !L->have_ktimers) {
        for (auto& kt : L->ktimer)
            for (auto& ev : kt.ev) HIP_TRY(ctx, hipEventCreate(&ev));
        L->have_ktimers = true;
    }
    struct TimerScope {  // whatever path leaves this function, the thread's launches are plain again
        ~TimerScope() { g_kernel_timer = nullptr; }
    } timer_scope;
    if (timing == 2)
        for (auto& kt : L->ktimer) kt.used = 0;
    // mark(i): stage i - 1 ends here and stage i begins
    auto mark = [&](int i) -> hipError_t {
        if (timing == 2) g_kernel_timer = i < RBMOE_NUM_STAGES - 1 ? &L->ktimer[i] : nullptr;
        return timing == 1 ? hipEventRecord(L->ev[i], s) : hipSuccess;
    };
    HIP_TRY(ctx, mark(0));

    const bool mfma = L->use_stream;
    const bool f32mc = L->use_f32_mc;
    // (training, which may still be switched on before the weights are set: no gain from tall tiles where gate/up also stores the
    // pre-activations, and the backward takes this table; padding: fewer rows than are counted here)
    const bool for_training = L->training || !L->weights_set;
    const int tile_m0 = mfma ? (for_training || valid ? kStreamTileM : stream_tile_m(T * k, E, F, d))
                             : (L->f32_rows ? f32_tile_m(T * k, E) : kGenericTileM);
    L->last_tile_m = tile_m0;
    L->kernel_name = mfma ? (wk == WeightKind::I8 ? "mfma_bf16_stream_int8w" : "mfma_bf16_stream")
                          : (f32mc ? "mfma_f32" : "generic");
    // a training layer keeps the gathered rows: the weight gradients of gate and up multiply by them
    const bool gather_in_product = (mfma || L->f32_rows) && !L->explicit_gather && !L->training;

    // whether the single-workgroup routing kernel would stage this call's rows in LDS: only then can it apply the
    // norm and write the bf16 copy of f32 rows
    const bool stages_rows = small_route_stages_rows(x, (const float*)L->router.p, T, d, E, abf) &&
                             (!norm_src || small_route_stages_rows(norm_src, (const float*)L->router.p, T, d, E, abf));
    const bool small = mfma && L->decode_path && !L->training && small_route_ok(T, E, k) && decode_shape_ok(F, d) &&
                       decode_shape_ok(d, F) && (!c.shared_expert || (decode_shape_ok(Fs, d) && decode_shape_ok(d, Fs)));
    RouterArgs ra{norm_src ? norm_src : x, (const float*)L->router.p, router_bias, valid, T, d, E, k,
                  (float*)L->P.p, (float*)L->lse.p, (int*)L->expert_of.p, (float*)L->gate_of.p,
                  (int*)L->rank_in_block.p, (int*)L->blockcnt.p, (float*)L->partial.p};
    if (cast) ra.rows16 = L->x16.p;
    ra.allow_fused = L->fused_router;
    ra.arrive = (int*)L->cmbcnt.p;
    if (L->tight) ra.min_tokens = kRouterTokens;
    ra.exact = L->router_exact;
    ra.exact_now = (const int*)L->cmbcnt.p + kRouterExactWord;
    if (L->router_q8) {
        ra.exact_now = nullptr;
        ra.wq = (const int8_t*)L->router_q.p;
        ra.wscale = (const float*)L->router_s.p;
    }
    if (norm_src) {
        ra.norm_w = (const float*)L->norm_w.p;
        ra.norm_eps = L->norm_eps;
        ra.xn_out = L->xn.p;
    }
    // the routing beside the gate/up products, in one launch
    bool front = small && L->decode_front && L->hall.p != nullptr && decode_front_ok(ra, abf) &&
                 (!L->router_q8 || wk == WeightKind::I8) && decode_front_pays(L, T, stages_rows, norm_src != nullptr);
    // (a caller without allocations, or one who switched the combined launch off, asked for these kernels by name)
    const bool choose = !static_scratch && L->decode_front;
    const bool batch = choose && small &&
                       (front ? !decode_front_beats_batch(L, T) : !decode_alone_beats_batch(L, T, stages_rows));
    if (batch) front = false;
    if (static_scratch && front && carve_decode_work(L, T, true, nullptr, nullptr) > (size_t)RBMOE_STATIC_SCRATCH_BYTES)
        front = false;
    // (without it a quantized router takes the large-batch sequence)
    const bool decode_ok = small && !batch && (front || (!L->router_q8 && (!cast || stages_rows)));
    const bool norm_in_route = norm_src && decode_ok && (front || stages_rows);
    Work wk_ = work_of_layer(L);
    if (static_scratch) {
        if (!decode_ok) {
            char buf[200];
            std::snprintf(buf, sizeof buf,
                          "rbmoe_forward_static takes decode-shaped calls only: 1 to %d tokens of a layer with bf16 or "
                          "int8 weights on the matrix-core path, not in training mode (got %d tokens)",
                          kSmallRouteMaxTokens, T);
            return fail(ctx, RBMOE_UNSUPPORTED, buf);
        }
        const size_t need = carve_decode_work(L, T, front, nullptr, nullptr);
        if (need > (size_t)RBMOE_STATIC_SCRATCH_BYTES) {
            char buf[200];
            std::snprintf(buf, sizeof buf, "this call needs %zu bytes of scratch, the static buffer holds %zu", need,
                          (size_t)RBMOE_STATIC_SCRATCH_BYTES);
            return fail(ctx, RBMOE_UNSUPPORTED, buf);
        }
        // Nothing of it is cleared: every word a kernel of this call reads was written by an earlier kernel of
        // the same call (the tile-table entries past *ntiles, which the product kernels fetch and drop, may be
        // a previous call's).
        carve_decode_work(L, T, front, static_cast<unsigned char*>(static_scratch), &wk_);
    }
    // the rows the expert products read
    const void* xe = cast ? wk_.x16 : x;
    const RouterArgs front_args = ra;  // (the routing beside the products has its own way with the norm)
    bool norm_apart = false;           // the norm runs by itself
    const RouterPlan rplan = plan_router_behind_norm(ra, x, abf, &norm_apart);
    const bool cast_apart = cast && L->router_q8 && !rplan.q8_writes_rows16;
    if (cast_apart) ra.rows16 = nullptr;
    if (decode_ok ? norm_src && !norm_in_route : norm_apart)
        HIP_TRY(ctx, launch_rmsnorm(norm_src, (const float*)L->norm_w.p, L->norm_eps, T, d, L->xn.p, abf, s));

    // ---- a few tokens: route in one workgroup, then stream the touched weights once -------
    if (decode_ok) {
        L->kernel_name = front ? (wk == WeightKind::I8 ? "mfma_bf16_decode_front_int8w" : "mfma_bf16_decode_front")
                               : (wk == WeightKind::I8 ? "mfma_bf16_decode_int8w" : "mfma_bf16_decode");
        SmallRouteArgs sr{};
        sr.x = x; sr.wr = (const float*)L->router.p; sr.bias = router_bias; sr.valid = valid;
        if (norm_in_route) {
            sr.x = norm_src; sr.norm_w = (const float*)L->norm_w.p; sr.norm_eps = L->norm_eps; sr.xn_out = L->xn.p;
        }
        if (cast) sr.rows16 = wk_.x16;
        sr.T = T; sr.d = d; sr.E = E; sr.k = k;
        sr.w_aux = c.aux_loss_weight; sr.w_z = c.router_z_loss_weight;
        sr.tile_m = kDecodeTileM;
        sr.P = wk_.P; sr.lse = wk_.lse;
        sr.expert_of = wk_.expert_of; sr.gate_of = wk_.gate_of;
        sr.counts = wk_.counts; sr.offsets = wk_.offsets;
        sr.tile_expert = wk_.tile_expert; sr.tile_row0 = wk_.tile_row0; sr.tile_rows = wk_.tile_rows;
        sr.ntiles = wk_.ntiles; sr.losses = wk_.losses;
        sr.perm_slot = wk_.perm_slot; sr.perm_token = wk_.perm_token; sr.inv_pos = wk_.inv_pos;
        for (auto& r : L->replay) r = nullptr;
        if (!front) {
            HIP_TRY(ctx, launch_route_small(sr, abf, s));
            L->replay[RBMOE_STAGE_ROUTER] = [=](hipStream_t st) { return launch_route_small(sr, abf, st); };
        }
        HIP_TRY(ctx, mark(1));
        HIP_TRY(ctx, mark(2));
        HIP_TRY(ctx, mark(3));

        DecodeGemmArgs d1{};
        d1.a = xe; d1.row_index = wk_.perm_token;
        d1.w = L->wgu.p; d1.w_expert_stride = (size_t)2 * F * d;
        d1.scales = wk == WeightKind::I8 ? (const float*)L->sgu.p : nullptr; d1.s_expert_stride = (size_t)2 * F;
        d1.N = F; d1.K = d;
        d1.tile_expert = wk_.tile_expert; d1.tile_row0 = wk_.tile_row0;
        d1.tile_rows = wk_.tile_rows; d1.ntiles = wk_.ntiles;
        d1.max_tiles = (T * k) / kDecodeTileM + E;
        d1.out = wk_.h;
        d1.swiglu = 1;
        if (c.shared_expert) {
            d1.a_shared = xe; d1.w_shared = L->swgu.p;
            d1.scales_shared = wk == WeightKind::I8 ? (const float*)L->ssgu.p : nullptr;
            d1.N_shared = Fs; d1.K_shared = d; d1.T_shared = T; d1.out_shared = wk_.hs;
        }
        DecodeLayoutArgs lay{wk_.P, wk_.lse, wk_.expert_of, valid, T, E, k, c.aux_loss_weight, c.router_z_loss_weight,
                             wk_.counts, wk_.offsets, wk_.tile_expert, wk_.tile_row0, wk_.tile_rows, wk_.ntiles, wk_.losses,
                             wk_.perm_slot, wk_.perm_token, wk_.inv_pos};
        if (front) {
            RouterArgs fr = front_args;  // (the products read the same rows: raw ones in front of a norm, f32 ones as they are)
            fr.P = wk_.P; fr.lse = wk_.lse; fr.expert_of = wk_.expert_of; fr.gate_of = wk_.gate_of;
            d1.a = fr.x;
            if (c.shared_expert) d1.a_shared = fr.x;
            d1.row_index = nullptr;
            d1.out = wk_.hall;
            HIP_TRY(ctx, launch_decode_front(fr, d1, abf, wk, s));
            L->replay[RBMOE_STAGE_GATE_UP] = [=](hipStream_t st) { return launch_decode_front(fr, d1, abf, wk, st); };
        } else {
            HIP_TRY(ctx, launch_decode_gemm(d1, wk, s));
            L->replay[RBMOE_STAGE_GATE_UP] = [=](hipStream_t st) { return launch_decode_gemm(d1, wk, st); };
        }
        HIP_TRY(ctx, mark(4));

        DecodeGemmArgs d2 = d1;
        d2.a = wk_.h; d2.row_index = nullptr;
        if (front) {  // the routed rows are picked out of the per-expert hidden rows: row token of expert e
            d2.a = wk_.hall; d2.row_index = wk_.perm_token; d2.a_expert_rows = T;
        }
        d2.w = L->wd.p; d2.w_expert_stride = (size_t)d * F;
        d2.scales = wk == WeightKind::I8 ? (const float*)L->sd.p : nullptr; d2.s_expert_stride = (size_t)d;
        d2.N = d; d2.K = F;
        d2.out = wk_.y;
        d2.swiglu = 0;
        if (c.shared_expert) {
            d2.a_shared = wk_.hs; d2.w_shared = L->swd.p;
            d2.scales_shared = wk == WeightKind::I8 ? (const float*)L->ssd.p : nullptr;
            d2.N_shared = d; d2.K_shared = Fs; d2.out_shared = wk_.ys;
        }
        // the combine inside the same launch: the last workgroup of every block of 32 output columns to finish
        // sums that block (same order, same roundings as combine_vec_kernel)
        const bool fold = L->decode_fold && d / 32 <= kDecodeCombineMaxBlocks && wk_.cmb_counter != nullptr;
        if (fold) {
            d2.cmb_counter = wk_.cmb_counter;
            d2.cmb_inv_pos = wk_.inv_pos; d2.cmb_gate_of = wk_.gate_of;
            d2.cmb_residual = residual; d2.cmb_out = out;
            d2.cmb_T = T; d2.cmb_k = k; d2.cmb_f32 = abf ? 0 : 1;
        }
        // behind the routing-beside-the-products launch the down launch has one row of workgroups per expert, whose weights
        // go out before anything of the routing is read, and makes the tables beside them; with a row or two, a workgroup
        // takes all rows of its columns (`few`)
        const bool by_expert = front && fold && L->decode_down_by_expert && decode_down_by_expert_ok(d2, E, T, k);
        const bool few = fold && L->decode_down_by_expert && decode_down_few_ok(d2, wk, T, k);
        if (few) {
            HIP_TRY(ctx, launch_decode_down_few(d2, lay, wk, s));
            L->replay[RBMOE_STAGE_DOWN] = [=](hipStream_t st) { return launch_decode_down_few(d2, lay, wk, st); };
        } else if (by_expert) {
            HIP_TRY(ctx, launch_decode_down_by_expert(d2, lay, wk, s));
            L->replay[RBMOE_STAGE_DOWN] = [=](hipStream_t st) { return launch_decode_down_by_expert(d2, lay, wk, st); };
        } else {
            if (front) HIP_TRY(ctx, launch_decode_layout(lay, s));
            HIP_TRY(ctx, launch_decode_gemm(d2, wk, s));
            L->replay[RBMOE_STAGE_DOWN] = [=](hipStream_t st) { return launch_decode_gemm(d2, wk, st); };
        }
        if (L->record_routed) HIP_TRY(ctx, hipEventRecord(L->record_routed, s));
        HIP_TRY(ctx, mark(5));
        HIP_TRY(ctx, mark(6));
        if (!fold) {
            CombineArgs cd{wk_.y, c.shared_expert ? wk_.ys : nullptr, residual, wk_.inv_pos, wk_.gate_of, T, d, k, out};
            cd.rows_bf16 = cast;
            HIP_TRY(ctx, launch_combine(cd, abf, s));
            L->replay[RBMOE_STAGE_COMBINE] = [=](hipStream_t st) { return launch_combine(cd, abf, st); };
        }
        HIP_TRY(ctx, mark(7));
        L->last_T = T;
        L->last = wk_;
        L->last_front = front;
        L->last_parts = 1;
        L->last_few = few;
        L->last_by_slot = front && (few || by_expert);
        L->x_saved = nullptr;
        return RBMOE_OK;
    }

    // MoeCache keeps the input (src/moe.rs:133-135).  Behind the norm the input is the layer's own buffer of normed rows,
    // which nothing writes before the next forward of the layer.
    L->x_saved = norm_src ? L->xn.p : L->xc.p;
    if (L->training && T > 0 && !norm_src)
        HIP_TRY(ctx, hipMemcpyAsync(L->xc.p, x, (size_t)T * d * dtype_size(c.act_dtype), hipMemcpyDeviceToDevice, s));

    if ((mfma || f32mc) && !cast && T > 0 && !starts_on_piece(x)) {
        if (!L->training)
            HIP_TRY(ctx, hipMemcpyAsync(L->st_x.p, x, (size_t)T * d * dtype_size(c.act_dtype), hipMemcpyDeviceToDevice, s));
        xe = L->training ? L->xc.p : L->st_x.p;
    }

    for (auto& r : L->replay) r = nullptr;
    auto run_on = [=](const GroupedArgs& g, hipStream_t st) -> hipError_t {
        if (mfma) return launch_grouped_stream(g, wk, st);
        if (L->f32_rows) return launch_grouped_f32(g, wk, st);
        return launch_grouped_generic(g, abf, wk, kGenericTileM, st);
    };
    auto run = [&](const GroupedArgs& g, bool) -> hipError_t { return run_on(g, s); };
    // The shared expert (src/moe.rs:313-319) takes every row and needs nothing of the routing: its products run in the
    // routed experts' launches, or with a second stream beside the routing kernels, which are bound by the vector units
    // and by latency and leave the matrix cores idle.  (Neither when the stages are timed one by one; not beside over f32
    // rows, whose bf16 copy the logits kernel has yet to write.)
    GroupedArgs s1{};  // gate/up, and (s2) the down product
    s1.a = xe;
    s1.w = L->swgu.p;
    s1.scales = wk == WeightKind::I8 ? (const float*)L->ssgu.p : nullptr;
    s1.N = Fs;
    s1.K = d;
    s1.dense_rows = T;
    s1.out = L->hs.p;
    s1.swiglu = true;
    s1.group_m = L->group_m;
    if (L->training) s1.gu_out = L->gus.p;
    GroupedArgs s2 = s1;
    s2.a = L->hs.p;
    s2.w = L->swd.p;
    s2.scales = wk == WeightKind::I8 ? (const float*)L->ssd.p : nullptr;
    s2.gu_out = nullptr;
    s2.N = d;
    s2.K = Fs;
    s2.out = L->ys.p;
    s2.swiglu = false;
    if (L->group_m == 0) s2.group_m = 4;
    auto shared_expert = [&](hipStream_t st) -> hipError_t {
        const hipError_t e = run_on(s1, st);
        return e != hipSuccess ? e : run_on(s2, st);
    };
    // Its tiles join the routed experts' launches where those do not fill the chip: below 1024 rows, where the products
    // would otherwise follow one another, and up to kSharedInsideTiles gate/up tiles in all.  Above, it runs beside the
    // routing kernels.  us a step, inside against beside (one behind the other below 1024 rows), at so many tiles: d 512,
    // 8 experts of 352 and one shared, 64 rows 33.6 / 46.3, 2048 rows (168 tiles) 42.5 / 63.4, 4096 (312) 56.1 / 66.3, 8192
    // (600) 79.6 / 86.2; d 768, 8 of 1408, 256 rows 43.2 / 63.2, 2048 (616) 76.5 / 80.4, 4096 (1144) 112.0 / 111.2; d 1024,
    // 64 of 704, six a row, 1000 rows 126.5 / 139.0, 2048 (1136) 164.5 / 154.0.
    constexpr int kSharedInsideTiles = 768;
    const int gate_up_tiles = ((T * k) / kStreamTileM + E) * ((F + 127) / 128) + (T + 127) / 128 * ((Fs + 127) / 128);
    // Over f32 rows (their kernels have tiles of 64 x 128 where a launch is large) the same below 1024 rows, and up to 400 such
    // tiles: us a step, inside / one behind the other (from 1024 rows on beside), d 512, 8 of 352, bf16 weights, 4 rows 32.6 /
    // 44.1, 512 39.2 / 49.7, 1024 (156 tiles) 45.8 / 61.2, 2048 (300) 63.1 / 72.0; f32 weights, 200 rows 35.2 / 50.3, 2048 84.1 / 83.0,
    // 4096 (588) 132.7 / 127.5; d 1024, 4 of 910, 24 rows 46.5 / 70.0, 1024 (272) 114.0 / 114.1, 2048 (528) 188.7 / 177.2; d 768,
    // 8 of 1408, 512 rows 111 / 123, 1024 (572) 179 / 158.
    constexpr int kSharedInsideF32Tiles = 400;
    const int f32_tiles = ((T * k) / 64 + (E + 1) / 2) * ((F + 127) / 128) + (T + 63) / 64 * ((Fs + 127) / 128);
    const bool shared_joins = c.shared_expert && T > 0 &&
                              (mfma ? T < 1024 || gate_up_tiles <= kSharedInsideTiles
                                    : L->f32_rows && f32_joins(F, Fs) && (T < 1024 || f32_tiles <= kSharedInsideF32Tiles));
    const bool shared_inside = shared_joins && !timed;
    auto with_shared = [&](GroupedArgs g, const GroupedArgs& sh) {
        g.dense2 = {sh.a, sh.w, sh.scales, sh.N, sh.K, sh.dense_rows, sh.out, sh.gu_out};
        return g;
    };
    struct JoinGuard {  // an error between fork and join must not leave the side stream forked (a capture could not end)
        rbmoe_ctx* ctx;
        hipStream_t main;
        bool armed = false;
        ~JoinGuard() {
            if (armed) (void)hipStreamWaitEvent(main, ctx->ev_join, 0);
        }
    } join_guard{ctx, s};
    bool shared_forked = false;
    auto fork_shared = [&]() -> int {
        if (c.shared_expert && !shared_inside && T >= 1024 && !timed && !cast && L->shared_beside && (mfma || L->f32_rows) &&
            ensure_side_stream(ctx) == RBMOE_OK) {
            HIP_TRY(ctx, hipEventRecord(ctx->ev_fork, s));
            HIP_TRY(ctx, hipStreamWaitEvent(ctx->side_stream, ctx->ev_fork, 0));
            const hipError_t e = shared_expert(ctx->side_stream);
            (void)hipEventRecord(ctx->ev_join, ctx->side_stream);  // recorded whatever happened: the join below always works
            join_guard.armed = true;
            shared_forked = true;
            if (e != hipSuccess) return hip_fail(ctx, e, "shared expert on the side stream");
        }
        return RBMOE_OK;
    };
    // (rows that the router's launch norms on its way are not there before it)
    const bool shared_first = ra.norm_w == nullptr;
    if (shared_first)
        if (const int rc = fork_shared()) return rc;

    if (cast_apart)
        HIP_TRY(ctx, launch_cast_rows_bf16((const float*)x, L->x16.p, (long long)T * d, s));
    HIP_TRY(ctx, launch_router(ra, rplan, abf, s));
    if (!shared_first)
        if (const int rc = fork_shared()) return rc;
    RouterArgs again = ra;  // (the rows are normed by now; in an in-place block step the raw ones are gone)
    if (again.norm_w) {
        again.x = x;
        again.norm_w = nullptr;
        again.xn_out = nullptr;
    }
    // (the same tokens a block with the norm and without: a norm that costs tokens is not taken along)
    const RouterPlan again_plan = plan_router(again, abf);
    if (again_plan.block_tokens == rplan.block_tokens)
        L->replay[RBMOE_STAGE_ROUTER] = [=](hipStream_t st) { return launch_router(again, again_plan, abf, st); };
    HIP_TRY(ctx, mark(1));

    HIP_TRY(ctx, mark(2));  // an interval with no work in it: the cost of one pair of event records

    DispatchArgs da{};
    da.x = xe;
    da.expert_of = (const int*)L->expert_of.p;
    da.rank_in_block = (const int*)L->rank_in_block.p;
    da.blockcnt = (const int*)L->blockcnt.p;
    da.partial = (const float*)L->partial.p;
    da.blockbase = (int*)L->blockbase.p;
    da.T = T; da.d = d; da.E = E; da.k = k;
    da.block_tokens = rplan.block_tokens;
    da.w_aux = c.aux_loss_weight; da.w_z = c.router_z_loss_weight;
    da.tile_m = tile_m0;
    da.counts = (int*)L->counts.p; da.offsets = (int*)L->offsets.p;
    da.tile_expert = (int*)L->tile_expert.p; da.tile_row0 = (int*)L->tile_row0.p; da.tile_rows = (int*)L->tile_rows.p;
    da.ntiles = (int*)L->ntiles.p; da.losses = (float*)L->losses.p;
    da.perm_slot = (int*)L->perm_slot.p; da.perm_token = (int*)L->perm_token.p; da.inv_pos = (int*)L->inv_pos.p;
    da.xg = gather_in_product ? nullptr : L->xg.p;
    GroupedArgs g1{};
    g1.a = gather_in_product ? xe : L->xg.p;
    g1.row_index = gather_in_product ? (const int*)L->perm_token.p : nullptr;
    g1.w = L->wgu.p;
    g1.w_expert_stride = (size_t)2 * F * d;
    g1.scales = wk == WeightKind::I8 ? (const float*)L->sgu.p : nullptr;
    g1.s_expert_stride = (size_t)2 * F;
    g1.N = F;
    g1.K = d;
    g1.tile_expert = (const int*)L->tile_expert.p;
    g1.tile_row0 = (const int*)L->tile_row0.p;
    g1.tile_rows = (const int*)L->tile_rows.p;
    g1.ntiles = (const int*)L->ntiles.p;
    g1.max_tiles = T > 0 ? (T * k) / tile_m0 + E : 0;
    g1.likely_tiles = likely_tiles(T * k, E, tile_m0);
    g1.tile_m = tile_m0;
    g1.routed_rows = T * k;
    g1.groups = E;
    g1.dense_rows = -1;
    g1.out = L->h.p;
    g1.swiglu = true;
    g1.group_m = L->group_m;
    if (L->training) g1.gu_out = L->gu.p;
    // No launch for the dispatch: the gate/up product works its tiles out by itself and writes the tables on the way.  The
    // launch and its chain (4 to 9 us) are saved, but every workgroup's own chain gets longer, so it pays for one round of
    // workgroups, two a compute unit.  us a forward, without / with the launch, at so many gate/up tiles: d 256, 4 experts of 704,
    // 40 rows 24.3 / 30.2, 8192 rows (396 tiles) 42.3 / 46.3; d 512, 8 experts of 352 and a shared one, 64 rows 26.8 / 30.9, 2048
    // (156) 37.1 / 40.7, 6144 (444) 71.2 / 76.3, 8192 (588) 86.2 / 85.0; d 768, 8 of 1408, 64 rows 33.0 / 37.3, 2048 (396) 58.8 / 62.8,
    // 4096 (748) 87.6 / 83.9; 16 of 1408, 512 rows 41.8 / 45.1, 3072 (616) 79.1 / 80.8, 8192 (1496) 151.0 / 139.4.
    // (Not where a host call fetches the tables beside the products, nor with events between the stages.)
    // Over f32 rows, workgroups as f32_workgroups counts them: d 512, 8 experts of 352 and a shared one, bf16 weights, 64 rows
    // 27.3 / 31.2, 1024 (600 workgroups) 42.6 / 45.8, 4096 (588) 91.0 / 93.0, 8192 (1164) 148.0 / 145.5; f32 weights, 8 of 1408, 1024
    // (396) 90.2 / 95.5, 4096 (1452) 260.7 / 261.6; d 768, 16 of 682, four a row, 512 (288) 91.9 / 95.2, 2048 (816) 205.5 / 202.8.
    constexpr int kDispatchInsideTiles = 512, kDispatchInsideF32 = 620;
    GroupedArgs first = shared_inside ? with_shared(g1, s1) : g1;
    const int workgroups = mfma ? g1.likely_tiles * ((F + 127) / 128) + (first.dense2.rows + 127) / 128 * ((first.dense2.N + 127) / 128)
                                : L->f32_rows ? f32_workgroups(first, wk) : 0;
    const bool dispatch_inside = (mfma || L->f32_rows) && gather_in_product && timing != 1 && !L->record_routed &&
                                 workgroups <= (mfma ? kDispatchInsideTiles : kDispatchInsideF32) && dispatch_in_product_ok(da);
    if (dispatch_inside) first.slots = routed_slots(da);
    if (!dispatch_inside) HIP_TRY(ctx, launch_dispatch(da, abf || cast, s));
    if (L->record_routed) HIP_TRY(ctx, hipEventRecord(L->record_routed, s));
    {
        const bool rows_bf16 = abf || cast;
        L->replay[RBMOE_STAGE_DISPATCH] = [=](hipStream_t st) { return launch_dispatch(da, rows_bf16, st); };
    }
    HIP_TRY(ctx, mark(3));
    HIP_TRY(ctx, run(first, true));
    L->replay[RBMOE_STAGE_GATE_UP] = [=](hipStream_t st) { return run_on(g1, st); };
    HIP_TRY(ctx, mark(4));

    GroupedArgs g2 = g1;
    g2.a = L->h.p;
    g2.gu_out = nullptr;
    g2.row_index = nullptr;
    g2.w = L->wd.p;
    g2.w_expert_stride = (size_t)d * F;
    g2.scales = wk == WeightKind::I8 ? (const float*)L->sd.p : nullptr;
    g2.s_expert_stride = (size_t)d;
    g2.N = d;
    g2.K = F;
    g2.out = L->y.p;
    g2.swiglu = false;
    // M-tiles that walk the column tiles together on one XCD: what they share must fit its 4 MiB L2 beside the
    // weights - eight tiles' token rows for the gate/up product (launch_grouped_stream's default), four tiles' hidden
    // rows, which are wider, for the down product (measured HBM-side traffic: 270 against 301 MB with groups of 8
    // against 4 for gate/up, 147 against 166 MB with 4 against 8 for down)
    if (L->group_m == 0) g2.group_m = 4;
    // The parts of the reduction are those of the call that is not timed, also where its shared expert has launches of its own here
    // and in the stage's replay, which is the routed experts' alone.
    const GroupedArgs call = shared_joins ? with_shared(g2, s2) : g2;
    if ((L->f32_rows || (mfma && d % 8 == 0)) && !for_training && T > 0 && d % 4 == 0 && k <= 8 &&
        (L->f32_rows || !c.shared_expert || shared_joins)) {
        g2.parts = mfma ? stream_parts(call) : f32_parts(call, wk);
        const size_t rows = (size_t)T * k + (shared_joins ? (size_t)T : 0);
        while (g2.parts > 1 && g2.parts * rows * d * 4 > parts_room(L)) g2.parts /= 2;
    }
    if (g2.parts > 1) {
        g2.out = static_cast<char*>(L->y.p) + parts_offset(L);
        g2.part_rows = T * k;
        wk_.y = g2.out;
        if (shared_joins) {
            s2.out = static_cast<float*>(g2.out) + (size_t)g2.parts * T * k * d;
            s2.parts = g2.parts;
            s2.part_rows = T;
        }
    }
    HIP_TRY(ctx, run(shared_inside ? with_shared(g2, s2) : g2, false));
    L->replay[RBMOE_STAGE_DOWN] = [=](hipStream_t st) { return run_on(g2, st); };
    HIP_TRY(ctx, mark(5));

    if (c.shared_expert && T > 0 && !shared_forked && !shared_inside) HIP_TRY(ctx, shared_expert(s));
    if (shared_forked) {
        HIP_TRY(ctx, hipStreamWaitEvent(s, ctx->ev_join, 0));
        join_guard.armed = false;
    }
    HIP_TRY(ctx, mark(6));

    CombineArgs ca{g2.out, c.shared_expert ? s2.out : nullptr, residual, (const int*)L->inv_pos.p,
                   (const float*)L->gate_of.p, T, d, k, out};
    ca.rows_bf16 = cast;
    ca.parts = g2.parts;
    ca.shared_in_parts = s2.parts > 1;
    ca.part_rows = g2.part_rows;
    HIP_TRY(ctx, launch_combine(ca, abf, s));
    L->replay[RBMOE_STAGE_COMBINE] = [=](hipStream_t st) { return launch_combine(ca, abf, st); };
    HIP_TRY(ctx, mark(7));
    L->last_T = T;
    L->last = wk_;
    L->last_parts = g2.parts;
    L->last_front = false;
    L->last_few = false;
    L->last_by_slot = false;
    return RBMOE_OK;
}

// Allocates and clears the buffers of `p` for a layer that already exists: the budget is checked before
// anything is allocated, and a failure part-way frees what this call had allocated, so that the layer is left as
// it was and the call can simply be made again.
int allocate_plan(rbmoe_layer* L, Plan& p, const char* what) {
    rbmoe_ctx* ctx = L->ctx;
    if (ctx->budget_bytes && ctx->allocated + p.total > ctx->budget_bytes) {
        char buf[200];
        std::snprintf(buf, sizeof buf, "memory budget exceeded: estimated %zu MiB exceeds budget %zu MiB",
                      (ctx->allocated + p.total + (1 << 20) - 1) >> 20, ctx->budget_bytes >> 20);
        return fail(ctx, RBMOE_MEMORY_BUDGET, buf);
    }
    size_t done = 0;
    hipError_t e = hipSetDevice(ctx->device);
    while (e == hipSuccess && done < p.items.size()) {
        auto& it = p.items[done];
        void* q = nullptr;
        e = hipMalloc(&q, it.second);
        if (e != hipSuccess) break;
        it.first->p = q;
        it.first->bytes = it.second;
        ctx->allocated += it.second;
        L->all.push_back(it.first);
        ++done;
        e = hipMemsetAsync(q, 0, it.second, ctx->stream);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e == hipSuccess) return RBMOE_OK;
    (void)hipGetLastError();
    (void)hipStreamSynchronize(ctx->stream);
    for (size_t i = 0; i < done; ++i) {
        Buf* b = p.items[i].first;
        (void)hipFree(b->p);
        if (ctx->allocated >= b->bytes) ctx->allocated -= b->bytes;
        b->p = nullptr;
        b->bytes = 0;
        for (size_t j = L->all.size(); j-- > 0;)
            if (L->all[j] == b) {
                L->all.erase(L->all.begin() + (long)j);
                break;
            }
    }
    if (e == hipErrorOutOfMemory)
        return fail(ctx, RBMOE_OUT_OF_MEMORY, std::string("out of memory while allocating ") + what);
    return hip_fail(ctx, e, what);
}

// f(), as it would come out for the tight layout.
template <typename F>
auto when_tight(rbmoe_layer* L, F&& f) {
    L->tight = true;
    choose_kernel_sets(L);
    auto r = f();
    L->tight = false;
    choose_kernel_sets(L);
    return r;
}

// allocate_plan of `make()`; where budget or memory refuse it and the layer can still give something back, the layer is
// made tight first.
template <typename F>
int allocate_or_tighten(rbmoe_layer* L, F&& make, const char* what) {
    rbmoe_ctx* ctx = L->ctx;
    {
        Plan p = make();
        const int rc = allocate_plan(L, p, what);
        if ((rc != RBMOE_MEMORY_BUDGET && rc != RBMOE_OUT_OF_MEMORY) || L->tight || L->weights_set || L->training) return rc;
        size_t held = 0;
        for (const auto& it : make_plan(L).items) held += it.first->bytes;
        const size_t needed = when_tight(L, [&] { return make_plan(L).total + make().total; });
        if (rc == RBMOE_MEMORY_BUDGET && ctx->allocated - held + needed > ctx->budget_bytes) return rc;
    }
    make_tight(L);
    Plan p = make();
    return allocate_plan(L, p, what);
}

// Buffers of the backward pass through the norm: allocated by whichever of rbmoe_set_feed_forward_norm and
// rbmoe_layer_enable_training comes second.
void add_block_training(rbmoe_layer* L, Plan& p) {
    if (!L->norm_w.p || L->xraw.p) return;
    const rbmoe_config& c = L->cfg;
    const size_t T = L->max_T, d = c.d_model, as = dtype_size(c.act_dtype);
    p.add(&L->xraw, T * d * as);
    p.add(&L->dxn, T * d * as);
    p.add(&L->inv_rms, T * 4);
    p.add(&L->norm_partial, (size_t)rmsnorm_grad_tiles((int)T) * d * 4);
    p.add(&L->g_norm, d * 4);
}
int ensure_block_training_buffers(rbmoe_layer* L) {
    if (!L->training || !L->norm_w.p || L->xraw.p) return RBMOE_OK;
    Plan p;
    add_block_training(L, p);
    return allocate_plan(L, p, "the norm's backward buffers");
}

Plan training_plan(rbmoe_layer* L) {
    const rbmoe_config& c = L->cfg;
    const size_t E = c.num_experts, d = c.d_model, F = L->Fw, Fs = L->Fsw, T = L->max_T, S = L->max_S;
    const size_t ws = dtype_size(c.weight_dtype);  // bytes per element of the transposed weight copies
    const size_t as = dtype_size(c.act_dtype);
    const size_t ps = L->cast_rows ? 2 : as;       // bytes per element of the rows the products read and write
    Plan p;
    p.add(&L->xc, T * d * as);
    if (L->cast_rows) p.add(&L->g16, T * d * 2);
    p.add(&L->gu, S * 2 * F * ps);
    p.add(&L->dy, S * d * ps);
    p.add(&L->dgu, S * 2 * F * ps);
    p.add(&L->dxg, S * d * ps);
    p.add(&L->grad_gates, S * 4);
    p.add(&L->ones, S * 4);
    p.add(&L->dlogits, T * E * 4);
    p.add(&L->dxr, T * d * as);
    p.add(&L->rpartial, (size_t)router_grad_chunks((int)T) * E * d * 4);
    p.add(&L->g_router, E * d * 4);
    p.add(&L->g_gu, E * 2 * F * d * 4);
    p.add(&L->g_down, E * d * F * 4);
    p.add(&L->wdT, E * F * d * ws);
    p.add(&L->wguT, E * d * 2 * F * ws);
    // (four tables: down and gate/up gradients of the routed experts and of the shared one)
    p.add(&L->wg_chunks, (size_t)4 * wgrad_table_ints(L) * 4);
    // How the weight gradients treat an expert far above the average share (and the shared expert, whose one
    // group of rows is always cut): in a fixed order by default (RBMOE_OPT_WGRAD_MODE for f32 atomics or no cut).
    if (L->wgrad_split == WgradSplit::Ordered) {
        const bool wbf = c.act_dtype == RBMOE_BF16 || L->cast_rows;
        // sized for every token count up to max_tokens: a smaller batch can need more partial matrices than the
        // largest one, because the cut limit follows the row count with a floor and a rounding
        const int k = c.experts_per_token;
        size_t need = std::max(weight_grad_partial_bytes_upto((int)d, (int)F, (int)E, false, (int)T, k, wbf),
                               weight_grad_partial_bytes_upto((int)(2 * F), (int)d, (int)E, false, (int)T, k, wbf));
        if (c.shared_expert)
            need = std::max(need, std::max(weight_grad_partial_bytes_upto((int)d, (int)Fs, 1, true, (int)T, 1, wbf),
                                           weight_grad_partial_bytes_upto((int)(2 * Fs), (int)d, 1, true, (int)T, 1, wbf)));
        p.add(&L->wg_partial, need);
    }
    p.add(&L->st_gout, T * d * as);
    p.add(&L->st_gin, T * d * as);
    if (c.shared_expert) {
        p.add(&L->gus, T * 2 * Fs * ps);
        p.add(&L->dgus, T * 2 * Fs * ps);
        p.add(&L->dxs, T * d * ps);
        p.add(&L->g_sgu, 2 * Fs * d * 4);
        p.add(&L->g_sdown, d * Fs * 4);
        p.add(&L->swdT, Fs * d * ws);
        p.add(&L->swguT, d * 2 * Fs * ws);
    }
    add_block_training(L, p);
    return p;
}

// The backward entry points differentiate the LAST forward, whose shape the reference takes from the cached input
// (src/moe.rs:349-350).  Here the cache is the layer's own state, so the caller states the shape of its buffers
// and a mismatch is refused before any of their bytes is read or written.
int backward_shape_problem(rbmoe_layer* L, int32_t tokens, int32_t cols) {
    rbmoe_ctx* ctx = L->ctx;
    char buf[160];
    if (cols != L->cfg.d_model) {
        std::snprintf(buf, sizeof buf, "gradient length %d does not match expected length %d", cols, L->cfg.d_model);
        return fail(ctx, RBMOE_INVALID_INPUT, buf);
    }
    if (tokens != L->last_T) {
        std::snprintf(buf, sizeof buf, "gradient rows %d do not match the %d rows of the last forward pass", tokens,
                      L->last_T);
        return fail(ctx, RBMOE_INVALID_INPUT, buf);
    }
    return RBMOE_OK;
}

// ---- host calls -----------------------------------------------------------------------------------------------
// Rows travel through pinned memory: a copy from pageable memory is cut into pieces that a host thread moves (and
// rounds, for f32 rows of a bf16 layer) while the DMA engine sends the pieces before; results go to the caller's
// memory directly when it is one of the library's pinned blocks.

// Bytes of a piece.  Every DMA costs about 8 us beside its bytes and the first piece's host copy is not covered by
// anything: 4.7 MB from pageable memory take 246 us in pieces of 256 KB, 174 in 512 KB, 148 in 1 MB, 143 in 1.5 MB,
// 163 in one (the link alone: 90).
constexpr size_t kCopyPiece = (size_t)1280 << 10;

// `n` elements of the caller's host array to the device; `stage` is room for them in the layer's element type.
int host_rows_in(rbmoe_ctx* ctx, void* dst, const void* src, size_t n, bool round_to_bf16, size_t es, unsigned char* stage,
                 bool stage_pinned, hipStream_t s) {
    if (n == 0) return RBMOE_OK;
    if (!round_to_bf16 && host_block_holds(src, n * es)) {
        HIP_TRY(ctx, hipMemcpyAsync(dst, src, n * es, hipMemcpyHostToDevice, s));
        return RBMOE_OK;
    }
    const size_t step = stage_pinned ? kCopyPiece / es : n;
    for (size_t i = 0; i < n; i += step) {
        const size_t m = std::min(step, n - i);
        if (round_to_bf16)
            host_rows_to_bf16(static_cast<const float*>(src) + i, reinterpret_cast<uint16_t*>(stage) + i, m);
        else
            std::memcpy(stage + i * es, static_cast<const unsigned char*>(src) + i * es, m * es);
        HIP_TRY(ctx, hipMemcpyAsync(static_cast<char*>(dst) + i * es, stage + i * es, m * es, hipMemcpyHostToDevice, s));
    }
    return RBMOE_OK;
}

// Device rows (`es` bytes an element) to the caller's array; what is left to do once the stream has come this far is
// noted in `po`.
int host_rows_out(rbmoe_ctx* ctx, const void* src, void* user, size_t n, bool widen_to_f32, size_t es, PendingOut& po,
                  hipStream_t s) {
    po.user = nullptr;
    po.from_bf16 = false;
    if (n == 0) return RBMOE_OK;
    const size_t out_bytes = n * (widen_to_f32 ? 4 : es);
    unsigned char* to = static_cast<unsigned char*>(user);
    bool pinned = host_block_holds(user, out_bytes);
    if (!pinned) {
        if (!po.out.take(out_bytes)) return fail(ctx, RBMOE_OUT_OF_MEMORY, "no host memory for the results");
        pinned = po.out.pinned();
        to = po.out.p;
        po.user = user;
    }
    po.elements = n;
    po.element_bytes = widen_to_f32 ? 4 : es;
    if (widen_to_f32 && pinned && n % 4 == 0 && reinterpret_cast<uintptr_t>(to) % 16 == 0) {
        HIP_TRY(ctx, launch_widen_rows(src, reinterpret_cast<float*>(to), n, s));
        return RBMOE_OK;
    }
    if (widen_to_f32) {  // bf16 rows to host memory of their own, widened by the host at the end
        if (po.user == nullptr) {
            if (!po.out.take(n * 2)) return fail(ctx, RBMOE_OUT_OF_MEMORY, "no host memory for the results");
            to = po.out.p;
            po.user = user;
        }
        po.from_bf16 = true;
    }
    HIP_TRY(ctx, hipMemcpyAsync(to, src, n * es, hipMemcpyDeviceToHost, s));
    return RBMOE_OK;
}

int host_out_finish(rbmoe_ctx* ctx, PendingOut& po) {
    if (!po.any) return RBMOE_OK;
    const hipError_t e = hipStreamSynchronize(po.stream);
    if (e == hipSuccess && po.user != nullptr) {
        if (po.from_bf16) host_rows_to_f32(reinterpret_cast<const uint16_t*>(po.out.p), static_cast<float*>(po.user), po.elements);
        else std::memcpy(po.user, po.out.p, po.elements * po.element_bytes);
    }
    po.any = false;
    po.user = nullptr;
    po.in.reset();
    po.out.reset();
    if (e != hipSuccess) return hip_fail(ctx, e, "hipStreamSynchronize");
    return RBMOE_OK;
}

int host_forward_finish(rbmoe_layer* L) { return host_out_finish(L->ctx, L->pending); }

// The routing tables of the last forward and its two losses to host memory, by one launch that writes them there
// (arrays outside the library's pinned blocks through `stage`).  The copies still to be made once the stream has come
// this far are left in `after`.
struct TableCopy {
    void* dst;
    const void* src;
    size_t bytes;
};
int fetch_tables(rbmoe_layer* L, const rbmoe_routing* r, float* losses, Staging& stage, std::vector<TableCopy>& after, hipStream_t s) {
    rbmoe_ctx* ctx = L->ctx;
    const int T = L->last_T, E = L->cfg.num_experts, k = L->cfg.experts_per_token;
    const size_t S = (size_t)T * k;
    const Work& w = L->last;
    struct Want {
        void* dst;
        const void* src;
        size_t words;
    } want[9];
    int nw = 0;
    auto add = [&](void* dst, const void* src, size_t words) {
        if (dst && words) want[nw++] = {dst, src, words};
    };
    if (r) {
        add(r->counts, w.counts, (size_t)E);
        add(r->offsets, w.offsets, (size_t)E + 1);
        add(r->expert_of, w.expert_of, S);
        add(r->gate_of, w.gate_of, S);
        add(r->perm_slot, w.perm_slot, S);
        add(r->perm_token, w.perm_token, S);
        add(r->probabilities, w.P, (size_t)T * E);
        add(r->log_sum_exp, w.lse, (size_t)T);
    }
    add(losses, w.losses, 2);
    size_t staged = 0;
    bool direct[9];
    for (int i = 0; i < nw; ++i) {
        direct[i] = reinterpret_cast<uintptr_t>(want[i].dst) % 4 == 0 && host_block_holds(want[i].dst, want[i].words * 4);
        if (!direct[i]) staged += want[i].words * 4;
    }
    if (staged && !stage.take(staged)) return fail(ctx, RBMOE_OUT_OF_MEMORY, "no host memory for the routing tables");
    CopySegment seg[kMaxCopySegments];
    int ns = 0;
    size_t at = 0;
    for (int i = 0; i < nw; ++i) {
        void* to = want[i].dst;
        if (!direct[i]) {
            to = stage.p + at;
            at += want[i].words * 4;
            after.push_back({want[i].dst, to, want[i].words * 4});
        }
        if (direct[i] || stage.pinned()) seg[ns++] = {want[i].src, to, (unsigned int)want[i].words};
        else HIP_TRY(ctx, hipMemcpyAsync(to, want[i].src, want[i].words * 4, hipMemcpyDeviceToHost, s));
    }
    HIP_TRY(ctx, launch_copy_segments(seg, ns, s));
    return RBMOE_OK;
}

// forward_train (or the block step) on host rows.  Returns when the routing tables and losses asked for are in place;
// `out` is complete after host_forward_finish.  `io`: dtype of x, residual and out, the layer's own or f32.
int host_forward_begin(rbmoe_layer* L, const void* x, int io, int T, int cols, const uint8_t* valid, const float* router_bias,
                       const void* residual, bool block, void* out, rbmoe_routing* routing, float* losses) {
    rbmoe_ctx* ctx = L->ctx;
    const rbmoe_config& c = L->cfg;
    if (const int rc = host_forward_finish(L)) return rc;  // (a call begun and never finished)
    if (block && !L->norm_set) return fail(ctx, RBMOE_INVALID_CONFIG, "the feed-forward norm has not been set");
    if (cols != c.d_model) {
        char buf[120];
        std::snprintf(buf, sizeof buf, "input length %d does not match expected length %d", cols, c.d_model);
        return fail(ctx, RBMOE_INVALID_INPUT, buf);
    }
    if (io != c.act_dtype && io != RBMOE_F32) return fail(ctx, RBMOE_INVALID_CONFIG, "rows must be f32 or the layer's own dtype");
    if (T < 0 || T > L->max_T) return fail(ctx, RBMOE_INVALID_INPUT, "token count outside [0, max_tokens]");
    if (T > 0 && (!x || !out)) return fail(ctx, RBMOE_NULL_POINTER, "x or out is NULL");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    const bool convert = io != c.act_dtype;  // f32 host rows of a bf16 layer
    const size_t as = dtype_size(c.act_dtype), n = (size_t)T * c.d_model, nbytes = n * as;
    hipStream_t s = ctx->stream;
    PendingOut& po = L->pending;
    struct Abandon {  // an error on the way: nothing may still be using the staging memory when it is given back
        rbmoe_ctx* ctx;
        PendingOut* po;
        ~Abandon() {
            if (!po) return;
            po->user = nullptr;
            (void)host_out_finish(ctx, *po);
        }
    } abandon{ctx, &po};
    po.any = true;
    po.stream = s;
    const size_t row_room = (nbytes + 255) & ~(size_t)255;
    const size_t res_at = row_room, valid_at = res_at + (residual ? row_room : 0), bias_at = valid_at + (((size_t)T + 255) & ~(size_t)255);
    if (!po.in.take(bias_at + (size_t)c.num_experts * 4)) return fail(ctx, RBMOE_OUT_OF_MEMORY, "no host memory for the rows");
    if (valid && T > 0) {
        std::memcpy(po.in.p + valid_at, valid, (size_t)T);
        HIP_TRY(ctx, hipMemcpyAsync(L->st_valid.p, po.in.p + valid_at, (size_t)T, hipMemcpyHostToDevice, s));
    }
    if (router_bias) {
        std::memcpy(po.in.p + bias_at, router_bias, (size_t)c.num_experts * 4);
        HIP_TRY(ctx, hipMemcpyAsync(L->st_bias.p, po.in.p + bias_at, (size_t)c.num_experts * 4, hipMemcpyHostToDevice, s));
    }
    if (const int rc = host_rows_in(ctx, L->st_x.p, x, n, convert, as, po.in.p, po.in.pinned(), s)) return rc;
    if (residual)
        if (const int rc = host_rows_in(ctx, L->st_res.p, residual, n, convert, as, po.in.p + res_at, po.in.pinned(), s)) return rc;
    const uint8_t* const dvalid = valid ? (const uint8_t*)L->st_valid.p : nullptr;
    const float* const dbias = router_bias ? (const float*)L->st_bias.p : nullptr;
    // the tables are fetched on the side stream, beside the expert products
    const bool tables = routing != nullptr || losses != nullptr;
    if (tables) {
        if (const int rc = ensure_side_stream(ctx)) return rc;
        L->record_routed = ctx->ev_routed;
    }
    int rc = block ? rbmoe_forward_block(L, L->st_x.p, T, cols, dvalid, dbias, L->st_out.p)
                   : forward_impl(L, L->st_x.p, T, cols, dvalid, dbias, residual ? L->st_res.p : nullptr, L->st_out.p, 0);
    L->record_routed = nullptr;
    if (rc != RBMOE_OK) return rc;
    Staging stage;
    std::vector<TableCopy> after;
    if (tables) {
        HIP_TRY(ctx, hipStreamWaitEvent(ctx->side_stream, ctx->ev_routed, 0));
        rc = fetch_tables(L, routing, losses, stage, after, ctx->side_stream);
        const hipError_t e = hipEventRecord(ctx->ev_fetched, ctx->side_stream);
        if (rc != RBMOE_OK || e != hipSuccess) {
            (void)hipStreamSynchronize(ctx->side_stream);
            return rc != RBMOE_OK ? rc : hip_fail(ctx, e, "hipEventRecord");
        }
    }
    rc = host_rows_out(ctx, L->st_out.p, out, n, convert, as, po, s);
    if (tables) {
        const hipError_t e = hipEventSynchronize(ctx->ev_fetched);
        if (rc == RBMOE_OK && e != hipSuccess) rc = hip_fail(ctx, e, "hipEventSynchronize");
        for (const TableCopy& t : after) std::memcpy(t.dst, t.src, t.bytes);
    }
    if (rc != RBMOE_OK) return rc;
    abandon.po = nullptr;
    return RBMOE_OK;
}

// backward (of the layer, or of the block step) on host gradients; `io` as in host_forward_begin.
int host_backward(rbmoe_layer* L, const void* grad_output, int io, int tokens, int cols, bool block, void* grad_input) {
    rbmoe_ctx* ctx = L->ctx;
    const rbmoe_config& c = L->cfg;
    if (!L->training) return fail(ctx, RBMOE_INVALID_CONFIG, "training is not enabled on this layer");
    if (block && !L->norm_set) return fail(ctx, RBMOE_INVALID_CONFIG, "the feed-forward norm has not been set");
    if (!block && L->last_T < 0) return fail(ctx, RBMOE_INVALID_INPUT, "no forward pass has run yet");
    if (block && (L->last_T < 0 || !L->last_was_block))
        return fail(ctx, RBMOE_INVALID_INPUT, "the last forward pass was not rbmoe_forward_block");
    if (const int rc = backward_shape_problem(L, tokens, cols)) return rc;  // before any byte of the buffers is touched
    if (io != c.act_dtype && io != RBMOE_F32) return fail(ctx, RBMOE_INVALID_CONFIG, "rows must be f32 or the layer's own dtype");
    const int T = L->last_T;
    if (T == 0) return RBMOE_OK;
    if (!grad_output || !grad_input) return fail(ctx, RBMOE_NULL_POINTER, "grad_output or grad_input is NULL");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    if (const int rc = host_forward_finish(L)) return rc;
    const bool convert = io != c.act_dtype;
    const size_t as = dtype_size(c.act_dtype), n = (size_t)T * c.d_model;
    hipStream_t s = ctx->stream;
    PendingOut po;
    po.any = true;
    po.stream = s;
    if (!po.in.take(n * as)) return fail(ctx, RBMOE_OUT_OF_MEMORY, "no host memory for the rows");
    int rc = host_rows_in(ctx, L->st_gout.p, grad_output, n, convert, as, po.in.p, po.in.pinned(), s);
    if (rc == RBMOE_OK)
        rc = block ? rbmoe_backward_block(L, L->st_gout.p, tokens, cols, L->st_gin.p)
                   : rbmoe_backward(L, L->st_gout.p, tokens, cols, L->st_gin.p);
    if (rc == RBMOE_OK) rc = host_rows_out(ctx, L->st_gin.p, grad_input, n, convert, as, po, s);
    if (rc != RBMOE_OK) po.user = nullptr;
    const int rc2 = host_out_finish(ctx, po);
    return rc != RBMOE_OK ? rc : rc2;
}

}  // namespace

extern "C" {

int rbmoe_forward(rbmoe_layer* L, const void* x, int32_t T, int32_t cols, const uint8_t* valid,
                  const float* router_bias, const void* residual, void* out) {
    return forward_impl(L, x, T, cols, valid, router_bias, residual, out, 0);
}

int rbmoe_forward_static(rbmoe_layer* L, const void* x, int32_t T, int32_t cols, const uint8_t* valid,
                         const float* router_bias, const void* residual, void* out) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    if (!L->ctx->static_scratch) return fail(L->ctx, RBMOE_DEVICE_ERROR, "the static scratch buffer was not resolved");
    return forward_impl(L, x, T, cols, valid, router_bias, residual, out, 0, nullptr, L->ctx->static_scratch);
}

int rbmoe_forward_timed(rbmoe_layer* L, const void* x, int32_t T, int32_t cols, const uint8_t* valid,
                        const float* router_bias, const void* residual, void* out, float* ms) {
    if (!ms) return fail(L ? L->ctx : nullptr, RBMOE_NULL_POINTER, "ms is NULL");
    int rc = forward_impl(L, x, T, cols, valid, router_bias, residual, out, 1);
    if (rc != RBMOE_OK) return rc;
    rbmoe_ctx* ctx = L->ctx;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    for (int i = 0; i < RBMOE_NUM_STAGES - 1; ++i)
        HIP_TRY(ctx, hipEventElapsedTime(&ms[i], L->ev[i], L->ev[i + 1]));
    HIP_TRY(ctx, hipEventElapsedTime(&ms[RBMOE_STAGE_TOTAL], L->ev[0], L->ev[RBMOE_NUM_STAGES - 1]));
    return RBMOE_OK;
}

int rbmoe_forward_kernel_times(rbmoe_layer* L, const void* x, int32_t T, int32_t cols, const uint8_t* valid,
                               const float* router_bias, const void* residual, void* out, float* ms) {
    if (!ms) return fail(L ? L->ctx : nullptr, RBMOE_NULL_POINTER, "ms is NULL");
    int rc = forward_impl(L, x, T, cols, valid, router_bias, residual, out, 2);
    if (rc != RBMOE_OK) return rc;
    rbmoe_ctx* ctx = L->ctx;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    float total = 0.0f;
    for (int i = 0; i < RBMOE_NUM_STAGES - 1; ++i) {
        ms[i] = 0.0f;
        for (int u = 0; u < L->ktimer[i].used; ++u) {
            float one = 0.0f;
            HIP_TRY(ctx, hipEventElapsedTime(&one, L->ktimer[i].ev[2 * u], L->ktimer[i].ev[2 * u + 1]));
            ms[i] += one;
        }
        total += ms[i];
    }
    ms[RBMOE_STAGE_TOTAL] = total;
    return RBMOE_OK;
}

int rbmoe_replay_stage(rbmoe_layer* L, int32_t stage, int32_t launches, float* ms_per_launch) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (stage < 0 || stage >= RBMOE_NUM_STAGES || launches <= 0)
        return fail(ctx, RBMOE_INVALID_INPUT, "stage out of range or launches not positive");
    if (L->last_T < 0) return fail(ctx, RBMOE_INVALID_INPUT, "no forward pass has run yet");
    if (!L->replay[stage]) return fail(ctx, RBMOE_UNSUPPORTED, "the last forward had no launch of its own for this stage");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    if (!ms_per_launch) {  // enqueue only: the caller times a sequence of its own
        for (int i = 0; i < launches; ++i) HIP_TRY(ctx, L->replay[stage](s));
        return RBMOE_OK;
    }
    if (!L->have_events) {
        for (auto& ev : L->ev) HIP_TRY(ctx, hipEventCreate(&ev));
        L->have_events = true;
    }
    HIP_TRY(ctx, L->replay[stage](s));  // warm-up: the stage's operands are back in the caches it usually finds them in
    HIP_TRY(ctx, hipEventRecord(L->ev[0], s));
    for (int i = 0; i < launches; ++i) HIP_TRY(ctx, L->replay[stage](s));
    HIP_TRY(ctx, hipEventRecord(L->ev[1], s));
    HIP_TRY(ctx, hipStreamSynchronize(s));
    float ms = 0.0f;
    HIP_TRY(ctx, hipEventElapsedTime(&ms, L->ev[0], L->ev[1]));
    *ms_per_launch = ms / (float)launches;
    return RBMOE_OK;
}

int rbmoe_forward_host(rbmoe_layer* L, const void* x, int32_t T, int32_t cols, const uint8_t* valid,
                       const float* router_bias, const void* residual, void* out) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    const int rc = host_forward_begin(L, x, L->cfg.act_dtype, T, cols, valid, router_bias, residual, false, out, nullptr, nullptr);
    return rc == RBMOE_OK ? host_forward_finish(L) : rc;
}

int rbmoe_forward_train_begin(rbmoe_layer* L, const void* x, int32_t x_dtype, int32_t T, int32_t cols, const uint8_t* valid,
                              const float* router_bias, const void* residual, int32_t block, void* out,
                              rbmoe_routing* routing, float* losses) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    return host_forward_begin(L, x, x_dtype, T, cols, valid, router_bias, residual, block != 0, out, routing, losses);
}

int rbmoe_forward_train_finish(rbmoe_layer* L) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    return host_forward_finish(L);
}

// ---------------------------------------------------------------------------
// The block's steps either side of the layer: RmsNorm::forward in front
// (src/norm.rs:41-61, src/transformer_block.rs:216), the residual add behind
// (src/transformer_block.rs:221-222).
// ---------------------------------------------------------------------------
int rbmoe_set_feed_forward_norm(rbmoe_layer* L, const float* weight, int32_t cols, float eps) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    const rbmoe_config& c = L->cfg;
    if (!weight) return fail(ctx, RBMOE_NULL_POINTER, "weight is NULL");
    if (cols != c.d_model) {
        char buf[120];
        std::snprintf(buf, sizeof buf, "norm weight length %d does not match expected length %d", cols, c.d_model);
        return fail(ctx, RBMOE_INVALID_INPUT, buf);
    }
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    if (!L->norm_w.p) {
        auto plan = [&] {
            Plan p;
            p.add(&L->xn, (size_t)L->max_T * c.d_model * dtype_size(c.act_dtype));
            p.add(&L->norm_w, (size_t)c.d_model * 4);
            return p;
        };
        if (const int rc = allocate_or_tighten(L, plan, "the normed rows")) return rc;
    }
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));  // no forward may still read the old weight
    HIP_TRY(ctx, hipMemcpy(L->norm_w.p, weight, (size_t)c.d_model * 4, hipMemcpyHostToDevice));
    L->norm_eps = eps;
    L->norm_set = true;
    return ensure_block_training_buffers(L);
}

int rbmoe_forward_block(rbmoe_layer* L, const void* x, int32_t T, int32_t cols, const uint8_t* valid,
                        const float* router_bias, void* out) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (!L->norm_set) return fail(ctx, RBMOE_INVALID_CONFIG, "the feed-forward norm has not been set");
    if (cols != L->cfg.d_model) {
        char buf[120];
        std::snprintf(buf, sizeof buf, "input length %d does not match expected length %d", cols, L->cfg.d_model);
        return fail(ctx, RBMOE_INVALID_INPUT, buf);
    }
    if (T < 0 || T > L->max_T) return fail(ctx, RBMOE_INVALID_INPUT, "token count outside [0, max_tokens]");
    if (T > 0 && (!x || !out)) return fail(ctx, RBMOE_NULL_POINTER, "x or out is NULL");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    if (L->training && T > 0)  // TransformerBlockCache keeps the residual (src/transformer_block.rs:224-232)
        HIP_TRY(ctx, hipMemcpyAsync(L->xraw.p, x, (size_t)T * cols * dtype_size(L->cfg.act_dtype),
                                    hipMemcpyDeviceToDevice, ctx->stream));
    const int rc = forward_impl(L, L->xn.p, T, cols, valid, router_bias, x, out, 0, x);
    if (rc == RBMOE_OK) L->last_was_block = true;
    return rc;
}

int rbmoe_forward_block_host(rbmoe_layer* L, const void* x, int32_t T, int32_t cols, const uint8_t* valid,
                             const float* router_bias, void* out) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    const int rc = host_forward_begin(L, x, L->cfg.act_dtype, T, cols, valid, router_bias, nullptr, true, out, nullptr, nullptr);
    return rc == RBMOE_OK ? host_forward_finish(L) : rc;
}

// ---------------------------------------------------------------------------
// Training: MoeLayer::backward (reference src/moe.rs:348-489).
// ---------------------------------------------------------------------------
int rbmoe_layer_enable_training(rbmoe_layer* L) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (L->training) return RBMOE_OK;
    const rbmoe_config& c = L->cfg;
    if (c.weight_dtype == RBMOE_I8)  // as in the reference: quantized experts are inference-only (src/ffn.rs:87-93)
        return fail(ctx, RBMOE_UNSUPPORTED, "the backward pass is not defined for int8 weights");
    if (L->weights_set)
        return fail(ctx, RBMOE_INVALID_CONFIG, "enable training before the weights are set");
    if (L->quantize_router)
        return fail(ctx, RBMOE_UNSUPPORTED, "the backward pass is not defined for a quantized router");
    // (f32 rows over bf16 weights - the reference's own mixed-precision shape, src/gpu_model.rs:2146-2153 - stay on
    // the matrix cores in both directions: the products read the bf16 copy of the rows that the forward writes
    // anyway and a bf16 copy of the upstream gradient that the backward pass writes first; the router's branch,
    // the norm and the sums that end in the caller's buffers stay f32)
    if (L->max_T > router_grad_max_tokens()) {  // found here, not in the middle of a backward pass
        char buf[160];
        std::snprintf(buf, sizeof buf, "the backward pass takes at most %d tokens a call, the layer was created for %d",
                      router_grad_max_tokens(), L->max_T);
        return fail(ctx, RBMOE_UNSUPPORTED, buf);
    }
    if (*training_widths_problem(L) && !L->tight && !*when_tight(L, [&] { return training_widths_problem(L); })) make_tight(L);
    if (const char* const problem = training_widths_problem(L); *problem) return fail(ctx, RBMOE_UNSUPPORTED, problem);
    // (the second stream first: a failure there must not leave buffers behind that a second attempt would allocate again)
    if (L->shared_beside)
        if (const int rc = ensure_side_stream(ctx)) return rc;
    if (const int rc = allocate_or_tighten(L, [&] { return training_plan(L); }, "the training buffers")) return rc;
    HIP_TRY(ctx, launch_fill_f32((float*)L->ones.p, 1.0f, (long long)L->max_S, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    L->side_branch = L->shared_beside;
    L->training = true;
    L->grads_clear = true;
    return RBMOE_OK;
}

int rbmoe_layer_set_option(rbmoe_layer* L, int32_t option, int32_t value) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    switch (option) {
        case RBMOE_OPT_FORCE_GENERIC:
            // the kernel set decides how the weights are laid out on the device
            if (L->weights_set || L->training)
                return fail(ctx, RBMOE_INVALID_CONFIG, "choose the kernel set before weights are set or training is enabled");
            L->force_generic = value != 0;
            choose_kernel_sets(L);
            return RBMOE_OK;
        case RBMOE_OPT_EXPLICIT_GATHER: L->explicit_gather = value != 0; return RBMOE_OK;
        case RBMOE_OPT_GROUP_M:
            if (value < 0) return fail(ctx, RBMOE_INVALID_CONFIG, "the group size must not be negative");
            L->group_m = value;
            return RBMOE_OK;
        case RBMOE_OPT_DECODE_PATH: L->decode_path = value != 0; return RBMOE_OK;
        case RBMOE_OPT_DECODE_FRONT: L->decode_front = value != 0; return RBMOE_OK;
        case RBMOE_OPT_FUSED_ROUTER: L->fused_router = value != 0; return RBMOE_OK;
        case RBMOE_OPT_DECODE_COMBINE_FOLD: L->decode_fold = value != 0; return RBMOE_OK;
        case RBMOE_OPT_DECODE_DOWN_BY_EXPERT: L->decode_down_by_expert = value != 0; return RBMOE_OK;
        case RBMOE_OPT_SIDE_STREAM:
            if (value != 0 && L->training)
                if (const int rc = ensure_side_stream(ctx)) return rc;
            L->shared_beside = value != 0;
            L->side_branch = value != 0;
            return RBMOE_OK;
        case RBMOE_OPT_WGRAD_MODE:
            if (value < 0 || value > 2) return fail(ctx, RBMOE_INVALID_CONFIG, "weight-gradient mode must be 0, 1 or 2");
            L->wgrad_split = value == 0 ? WgradSplit::Ordered : value == 1 ? WgradSplit::Atomic : WgradSplit::None;
            return RBMOE_OK;
        case RBMOE_OPT_WGRAD_GENERIC: L->wgrad_generic = value != 0; return RBMOE_OK;
        case RBMOE_OPT_QUANT_RULE:
            if (value != 0 && value != 1) return fail(ctx, RBMOE_INVALID_CONFIG, "the quantisation rule is 0 or 1");
            L->quant_rule = value;
            return RBMOE_OK;
        case RBMOE_OPT_QUANTIZE_ROUTER:
            if (value != 0 && L->training)
                return fail(ctx, RBMOE_UNSUPPORTED, "the backward pass is not defined for a quantized router");
            L->quantize_router = value != 0;
            return RBMOE_OK;
    }
    return fail(ctx, RBMOE_INVALID_CONFIG, "unknown option");
}

int rbmoe_zero_grads(rbmoe_layer* L) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (!L->training) return fail(ctx, RBMOE_INVALID_CONFIG, "training is not enabled on this layer");
    // The expert matrices (hundreds of MB) are not touched: they count as zero from here on, and the next
    // backward pass writes them instead of adding to them.  The router's gradient is small and is cleared.
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    // (a fill kernel, not a memset: a caller may capture a training step in a graph)
    HIP_TRY(ctx, launch_fill_f32((float*)L->g_router.p, 0.0f, (long long)(L->g_router.bytes / 4), ctx->stream));
    if (L->g_norm.p) HIP_TRY(ctx, launch_fill_f32((float*)L->g_norm.p, 0.0f, (long long)(L->g_norm.bytes / 4), ctx->stream));
    L->grads_clear = true;
    return RBMOE_OK;
}

int rbmoe_backward(rbmoe_layer* L, const void* grad_output, int32_t tokens, int32_t cols, void* grad_input) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (!L->training) return fail(ctx, RBMOE_INVALID_CONFIG, "training is not enabled on this layer");
    if (L->last_T < 0) return fail(ctx, RBMOE_INVALID_INPUT, "no forward pass has run yet");
    if (const int rc = backward_shape_problem(L, tokens, cols)) return rc;
    const rbmoe_config& c = L->cfg;
    const int E = c.num_experts, d = c.d_model, F = L->Fw, k = c.experts_per_token, Fs = L->Fsw, T = L->last_T;
    if (T == 0) return RBMOE_OK;
    if (!grad_output || !grad_input) return fail(ctx, RBMOE_NULL_POINTER, "grad_output or grad_input is NULL");
    // (a forward from before training mode has kept its rows only behind the norm)
    if (!L->x_saved) return fail(ctx, RBMOE_INVALID_INPUT, "no forward pass has run in training mode yet");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    const bool xbf = c.act_dtype == RBMOE_BF16;       // the caller's rows and gradients
    const bool cast = L->cast_rows;                   // ... are f32, the products' rows bf16
    const bool abf = xbf || cast;                     // the rows of the expert products
    const int S = T * k;
    const int* offsets = (const int*)L->offsets.p;
    const int* counts = (const int*)L->counts.p;
    // what the expert branch reads of the upstream gradient: the caller's rows, or their bf16 copy
    const void* gout = grad_output;
    if (cast) {
        HIP_TRY(ctx, launch_cast_rows_bf16((const float*)grad_output, L->g16.p, (long long)T * d, s));
        gout = L->g16.p;
    }

    if (!cast && c.shared_expert && (L->use_stream || L->use_f32_mc) && !starts_on_piece(grad_output)) {
        HIP_TRY(ctx, hipMemcpyAsync(L->st_gout.p, grad_output, (size_t)T * d * dtype_size(c.act_dtype), hipMemcpyDeviceToDevice, s));
        gout = L->st_gout.p;
    }

    // upstream of every expert: gate * dOut[token]; gate gradient: dOut[token] . Y[row]
    // (grad_gates of unrouted slots stays unwritten: the only reader skips padding rows)
    HIP_TRY(ctx, launch_scale_rows(gout, L->y.p, (const int*)L->perm_slot.p, (const int*)L->perm_token.p,
                                   (const float*)L->gate_of.p, offsets, E, d, S, L->dy.p, (float*)L->grad_gates.p, abf,
                                   s));
    // The router's branch needs nothing but the gate gradients from here on and is a handful of small launches
    // that leave most of the chip idle: it runs on the side stream, beside the products below, which meet
    // again at the final sum.  Gates -> probabilities -> logits with the two auxiliary losses
    // (src/moe.rs:421-478), then the router's weight and input gradients.
    const bool side = L->side_branch && ctx->side_stream != nullptr;
    const hipStream_t rs = side ? ctx->side_stream : s;
    if (side) {
        HIP_TRY(ctx, hipEventRecord(ctx->ev_fork, s));
        HIP_TRY(ctx, hipStreamWaitEvent(rs, ctx->ev_fork, 0));
    }
    // grad_input = sum over a token's slots of its expert rows + shared + router
    CombineArgs ca{L->dxg.p, c.shared_expert ? L->dxs.p : nullptr, L->dxr.p, (const int*)L->inv_pos.p,
                   (const float*)L->ones.p, T, d, k, grad_input};
    ca.rows_bf16 = cast;
    const bool combine_on_side = side && !c.shared_expert;
    const bool tables_early = side && !L->wgrad_generic;
    // From here to the join the side stream hangs off the main one: an error in between must not leave it forked
    // (a stream capture in progress could then never end), so the rest runs as one unit that is always joined.
    auto forked = [&]() -> int {
    if (tables_early) {
        // the chunk tables of the weight-gradient launches depend on nothing but the forward's counts and offsets:
        // they are worked out here, on the side stream, instead of in front of each product on the main one
        auto table = [&](int which, int M, int N, int groups, int dense_rows, int total_rows) -> hipError_t {
            if (!weight_grad_shape_ok(M, N, abf)) return hipSuccess;
            return launch_weight_grad(nullptr, M, nullptr, N, counts, offsets, groups, dense_rows, total_rows, L->wgrad_split,
                                      L->grads_clear, (int*)L->wg_chunks.p + (size_t)which * wgrad_table_ints(L),
                                      (float*)L->wg_partial.p, L->wg_partial.bytes, nullptr, 0, abf, rs, WgradPart::TableOnly);
        };
        HIP_TRY(ctx, table(0, d, F, E, -1, S));
        HIP_TRY(ctx, table(1, 2 * F, d, E, -1, S));
        if (c.shared_expert) {
            HIP_TRY(ctx, table(2, d, Fs, 1, T, T));
            HIP_TRY(ctx, table(3, 2 * Fs, d, 1, T, T));
        }
        HIP_TRY(ctx, hipEventRecord(ctx->ev_tables, rs));
    }
    HIP_TRY(ctx, launch_route_backward((const float*)L->P.p, (const float*)L->lse.p, (const int*)L->expert_of.p,
                                       (const float*)L->grad_gates.p, counts, offsets, T, E, k, c.aux_loss_weight,
                                       c.router_z_loss_weight, (float*)L->dlogits.p, rs));
    HIP_TRY(ctx, launch_router_grad((const float*)L->dlogits.p, L->x_saved, (const float*)L->router.p, T, d, E,
                                    (float*)L->rpartial.p, (float*)L->g_router.p, L->dxr.p, xbf, rs));

    // SwiGlu::backward over the routed rows (src/ffn.rs:87-120)
    GroupedArgs g{};
    g.tile_expert = (const int*)L->tile_expert.p;
    g.tile_row0 = (const int*)L->tile_row0.p;
    g.tile_rows = (const int*)L->tile_rows.p;
    g.ntiles = (const int*)L->ntiles.p;
    g.max_tiles = S / L->last_tile_m + E;  // the tile table of the last forward
    g.tile_m = L->last_tile_m;
    g.routed_rows = S;
    g.groups = E;
    g.dense_rows = -1;
    g.swiglu = false;
    g.group_m = L->group_m;
    GroupedArgs gh = g;  // grad_hidden = dY . Wdown
    gh.a = L->dy.p; gh.w = L->wdT.p; gh.w_expert_stride = (size_t)F * d; gh.N = F; gh.K = d;
    gh.swiglu_grad_gu = L->gu.p; gh.gu_out = L->dgu.p;  // the hidden gradient goes straight through SwiGLU's backward
    const WeightKind wk = c.weight_dtype == RBMOE_F32 ? WeightKind::F32 : WeightKind::BF16;
    auto prod_on = [&](const GroupedArgs& a, hipStream_t st) -> hipError_t {
        if (L->use_stream) return launch_grouped_stream(a, WeightKind::BF16, st);
        if (L->f32_rows) return launch_grouped_f32(a, wk, st);
        return launch_grouped_generic(a, abf, wk, kGenericTileM, st);
    };
    auto prod = [&](const GroupedArgs& a) -> hipError_t { return prod_on(a, s); };
    HIP_TRY(ctx, prod(gh));
    GroupedArgs gx = g;  // grad_input rows = dG . Wgate + dU . Wup
    gx.a = L->dgu.p; gx.w = L->wguT.p; gx.w_expert_stride = (size_t)d * 2 * F; gx.N = d; gx.K = 2 * F; gx.out = L->dxg.p;
    if (side) {
        // the input-gradient product follows the router's branch on the side stream, beside the weight gradients
        // (it needs dG | dU, which the launch above has just written)
        HIP_TRY(ctx, hipEventRecord(ctx->ev_fork2, s));
        HIP_TRY(ctx, hipStreamWaitEvent(rs, ctx->ev_fork2, 0));
        HIP_TRY(ctx, prod_on(gx, rs));
        // without a shared expert everything the final sum reads is written on the side stream: it runs there too,
        // beside the weight gradients
        if (combine_on_side) HIP_TRY(ctx, launch_combine(ca, xbf, rs));
        HIP_TRY(ctx, hipEventRecord(ctx->ev_join, rs));
    } else {
        HIP_TRY(ctx, prod(gx));
    }
    // weight gradients (src/param.rs:819-821): down += dY^T . H; (gate | up) += (dG | dU)^T . X[token]
    auto wgrad = [&](int table, const void* a, int M, const void* b, const int* b_rows, int N, int groups,
                     int dense_rows, int total_rows, float* out, size_t stride) -> hipError_t {
        if (!L->wgrad_generic && !b_rows && weight_grad_shape_ok(M, N, abf))
            return launch_weight_grad(a, M, b, N, counts, offsets, groups, dense_rows, total_rows,
                                      L->wgrad_split, L->grads_clear, (int*)L->wg_chunks.p + (size_t)table * wgrad_table_ints(L),
                                      (float*)L->wg_partial.p, L->wg_partial.bytes, out, stride, abf, s,
                                      tables_early ? WgradPart::ProductOnly : WgradPart::Both);
        if (L->grads_clear) {
            const hipError_t e = launch_fill_f32(out, 0.0f, (long long)((size_t)groups * (stride ? stride : (size_t)M * N)), s);
            if (e != hipSuccess) return e;
        }
        return launch_grouped_tn(a, M, b, b_rows, N, counts, offsets, groups, dense_rows, out, stride, abf, s);
    };
    if (tables_early) HIP_TRY(ctx, hipStreamWaitEvent(s, ctx->ev_tables, 0));
    HIP_TRY(ctx, wgrad(0, L->dy.p, d, L->h.p, nullptr, F, E, -1, S, (float*)L->g_down.p, (size_t)d * F));
    HIP_TRY(ctx, wgrad(1, L->dgu.p, 2 * F, L->xg.p, nullptr, d, E, -1, S, (float*)L->g_gu.p, (size_t)2 * F * d));
    // shared expert over every row (src/moe.rs:356-361)
    if (c.shared_expert) {
        GroupedArgs sh = g;
        sh.dense_rows = T;
        sh.a = gout; sh.w = L->swdT.p; sh.w_expert_stride = 0; sh.N = Fs; sh.K = d;
        sh.swiglu_grad_gu = L->gus.p; sh.gu_out = L->dgus.p;
        HIP_TRY(ctx, prod(sh));
        GroupedArgs sx = g;
        sx.dense_rows = T; sx.w_expert_stride = 0;
        sx.a = L->dgus.p; sx.w = L->swguT.p; sx.N = d; sx.K = 2 * Fs; sx.out = L->dxs.p;
        HIP_TRY(ctx, prod(sx));
        HIP_TRY(ctx, wgrad(2, gout, d, L->hs.p, nullptr, Fs, 1, T, T, (float*)L->g_sdown.p, 0));
        HIP_TRY(ctx, wgrad(3, L->dgus.p, 2 * Fs, cast ? L->x16.p : L->x_saved, nullptr, d, 1, T, T, (float*)L->g_sgu.p, 0));
    }
    // grad_input = sum over a token's slots of its expert rows + shared + router
    if (side) HIP_TRY(ctx, hipStreamWaitEvent(s, ctx->ev_join, 0));
    return RBMOE_OK;
    };
    const int rc = forked();
    if (rc != RBMOE_OK) {
        if (side) {  // rejoin whatever the side stream got to
            (void)hipEventRecord(ctx->ev_join, rs);
            (void)hipStreamWaitEvent(s, ctx->ev_join, 0);
        }
        return rc;
    }
    if (!combine_on_side) HIP_TRY(ctx, launch_combine(ca, xbf, s));
    L->grads_clear = false;
    return RBMOE_OK;
}

int rbmoe_backward_host(rbmoe_layer* L, const void* grad_output, int32_t tokens, int32_t cols, void* grad_input) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    return host_backward(L, grad_output, L->cfg.act_dtype, tokens, cols, false, grad_input);
}

int rbmoe_backward_train_host(rbmoe_layer* L, const void* grad_output, int32_t dtype, int32_t tokens, int32_t cols,
                              int32_t block, void* grad_input) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    return host_backward(L, grad_output, dtype, tokens, cols, block != 0, grad_input);
}

int rbmoe_backward_block(rbmoe_layer* L, const void* grad_output, int32_t tokens, int32_t cols, void* grad_input) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (!L->training) return fail(ctx, RBMOE_INVALID_CONFIG, "training is not enabled on this layer");
    if (!L->norm_set) return fail(ctx, RBMOE_INVALID_CONFIG, "the feed-forward norm has not been set");
    if (L->last_T < 0 || !L->last_was_block)
        return fail(ctx, RBMOE_INVALID_INPUT, "the last forward pass was not rbmoe_forward_block");
    if (const int rc = backward_shape_problem(L, tokens, cols)) return rc;
    const int T = L->last_T, d = L->cfg.d_model;
    if (T == 0) return RBMOE_OK;
    if (!grad_output || !grad_input) return fail(ctx, RBMOE_NULL_POINTER, "grad_output or grad_input is NULL");
    // grad_projected = feed_forward.backward(cache, grad_output)  (src/transformer_block.rs:257)
    const int rc = rbmoe_backward(L, grad_output, tokens, cols, L->dxn.p);
    if (rc != RBMOE_OK) return rc;
    // grad_residual = feed_forward_norm.backward(residual, grad_projected) + grad_output  (:258-263)
    HIP_TRY(ctx, launch_rmsnorm_backward(L->xraw.p, L->dxn.p, (const float*)L->norm_w.p, L->norm_eps, grad_output, T, d,
                                         grad_input, (float*)L->inv_rms.p, (float*)L->norm_partial.p,
                                         (float*)L->g_norm.p, L->cfg.act_dtype == RBMOE_BF16, ctx->stream));
    return RBMOE_OK;
}

int rbmoe_backward_block_host(rbmoe_layer* L, const void* grad_output, int32_t tokens, int32_t cols,
                              void* grad_input) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    return host_backward(L, grad_output, L->cfg.act_dtype, tokens, cols, true, grad_input);
}

int rbmoe_get_weight_grad(rbmoe_layer* L, int32_t which, int32_t expert, float* host, int32_t rows, int32_t cols) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (!L->training) return fail(ctx, RBMOE_INVALID_CONFIG, "training is not enabled on this layer");
    if (!host) return fail(ctx, RBMOE_NULL_POINTER, "host buffer is NULL");
    const rbmoe_config& c = L->cfg;
    const size_t E = c.num_experts, d = c.d_model, F = c.d_ff, Fs = L->Fs, Fw = L->Fw, Fsw = L->Fsw;
    const float* src = nullptr;
    size_t want_rows = 0, want_cols = 0, pitch = 0;  // pitch: of the rows in `src` where it is not want_cols
    const bool bad_expert = expert < 0 || (size_t)expert >= E;
    switch (which) {
        case RBMOE_W_ROUTER: src = (const float*)L->g_router.p; want_rows = E; want_cols = d; break;
        case RBMOE_W_GATE:
        case RBMOE_W_UP:
            if (bad_expert) return fail(ctx, RBMOE_INVALID_CONFIG, "expert index out of range");
            src = (const float*)L->g_gu.p + ((size_t)expert * 2 + (which == RBMOE_W_UP ? 1 : 0)) * Fw * d;
            want_rows = F; want_cols = d;
            break;
        case RBMOE_W_DOWN:
            if (bad_expert) return fail(ctx, RBMOE_INVALID_CONFIG, "expert index out of range");
            src = (const float*)L->g_down.p + (size_t)expert * d * Fw;
            want_rows = d; want_cols = F; pitch = Fw;
            break;
        case RBMOE_W_SHARED_GATE:
        case RBMOE_W_SHARED_UP:
            if (!c.shared_expert) return fail(ctx, RBMOE_INVALID_CONFIG, "the layer has no shared expert");
            src = (const float*)L->g_sgu.p + (size_t)(which == RBMOE_W_SHARED_UP ? 1 : 0) * Fsw * d;
            want_rows = Fs; want_cols = d;
            break;
        case RBMOE_W_SHARED_DOWN:
            if (!c.shared_expert) return fail(ctx, RBMOE_INVALID_CONFIG, "the layer has no shared expert");
            src = (const float*)L->g_sdown.p;
            want_rows = d; want_cols = Fs; pitch = Fsw;
            break;
        case RBMOE_W_NORM:
            if (!L->g_norm.p) return fail(ctx, RBMOE_INVALID_CONFIG, "the feed-forward norm has not been set");
            src = (const float*)L->g_norm.p;
            want_rows = 1; want_cols = d;
            break;
        default:
            return fail(ctx, RBMOE_INVALID_CONFIG, "unknown weight id");
    }
    if ((size_t)rows != want_rows || (size_t)cols != want_cols)
        return fail(ctx, RBMOE_INVALID_INPUT, "gradient shape does not match the weight");
    if (L->grads_clear && which != RBMOE_W_ROUTER && which != RBMOE_W_NORM) {  // cleared and not written since
        std::memset(host, 0, want_rows * want_cols * 4);
        return RBMOE_OK;
    }
    hipStream_t s = ctx->stream;
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    const size_t bytes = want_rows * want_cols * 4;
    if (pitch == 0) pitch = want_cols;
    if (host_block_holds(host, bytes) && reinterpret_cast<uintptr_t>(host) % 4 == 0) {
        // straight into the caller's pinned block, behind whatever the stream still has to do.  (Rows of a rounded width as a copy of
        // the runtime's, too: the stream's end is seen 3 to 5 us earlier behind one than behind a kernel that writes to host memory.  us
        // a training step over host matrices, such a kernel / this: 8 experts of 682, d 512, f32, 1000 rows 1604 / 1555, of 910, d 1024,
        // 150 rows 2383 / 2310.)
        if (pitch == want_cols) HIP_TRY(ctx, hipMemcpyAsync(host, src, bytes, hipMemcpyDeviceToHost, s));
        else HIP_TRY(ctx, hipMemcpy2DAsync(host, want_cols * 4, src, pitch * 4, want_cols * 4, want_rows, hipMemcpyDeviceToHost, s));
        HIP_TRY(ctx, hipStreamSynchronize(s));
        return RBMOE_OK;
    }
    if (pitch == want_cols) {
        HIP_TRY(ctx, hipStreamSynchronize(s));
        HIP_TRY(ctx, hipMemcpy(host, src, bytes, hipMemcpyDeviceToHost));
        return RBMOE_OK;
    }
    // Rows of a rounded width into memory of the caller's own: through a block of the pool, since a rectangular copy into plain memory
    // is a copy a row there, 7 us each.
    Staging stage;
    if (!stage.take(want_rows * pitch * 4)) return fail(ctx, RBMOE_OUT_OF_MEMORY, "no host memory for the gradient's rows");
    size_t apart = want_cols * 4;  // bytes from row to row of the block
    if (stage.pinned()) {
        HIP_TRY(ctx, hipMemcpy2DAsync(stage.p, apart, src, pitch * 4, apart, want_rows, hipMemcpyDeviceToHost, s));
    } else {
        apart = pitch * 4;
        HIP_TRY(ctx, hipMemcpyAsync(stage.p, src, want_rows * apart, hipMemcpyDeviceToHost, s));
    }
    HIP_TRY(ctx, hipStreamSynchronize(s));
    for (size_t r = 0; r < want_rows; ++r) std::memcpy(host + r * want_cols, stage.p + r * apart, want_cols * 4);
    return RBMOE_OK;
}

// Both getters: one launch on the context's stream, one wait.
static int get_tables(rbmoe_layer* L, const rbmoe_routing* r, float* losses) {
    rbmoe_ctx* ctx = L->ctx;
    if (L->last_T < 0) return fail(ctx, RBMOE_INVALID_INPUT, "no forward pass has run yet");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    Staging stage;
    std::vector<TableCopy> after;
    const int rc = fetch_tables(L, r, losses, stage, after, ctx->stream);
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    if (rc != RBMOE_OK) return rc;
    for (const TableCopy& t : after) std::memcpy(t.dst, t.src, t.bytes);
    return RBMOE_OK;
}

int rbmoe_get_losses(rbmoe_layer* L, float* aux_loss, float* z_loss) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    float v[2] = {0.f, 0.f};
    if (const int rc = get_tables(L, nullptr, v)) return rc;
    if (aux_loss) *aux_loss = v[0];
    if (z_loss) *z_loss = v[1];
    return RBMOE_OK;
}

int rbmoe_get_routing(rbmoe_layer* L, rbmoe_routing* r) {
    if (!L || !r) return fail(L ? L->ctx : nullptr, RBMOE_NULL_POINTER, "layer or routing is NULL");
    return get_tables(L, r, nullptr);
}

int rbmoe_get_expert_rows(rbmoe_layer* L, float* hidden, float* expert_out) {
    if (!L) return fail(nullptr, RBMOE_NULL_POINTER, "layer is NULL");
    rbmoe_ctx* ctx = L->ctx;
    if (L->last_T < 0) return fail(ctx, RBMOE_INVALID_INPUT, "no forward pass has run yet");
    const int E = L->cfg.num_experts, d = L->cfg.d_model, F = L->cfg.d_ff, Fw = L->Fw;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    int R = 0;
    HIP_TRY(ctx, hipMemcpy(&R, L->last.offsets + E, 4, hipMemcpyDeviceToHost));
    const bool abf = L->cfg.act_dtype == RBMOE_BF16 || L->cast_rows;  // the rows of a cast_rows layer are bf16
    auto fetch = [&](float* dst, const void* src, size_t n) -> int {
        if (!dst || n == 0) return RBMOE_OK;
        if (!abf) {
            HIP_TRY(ctx, hipMemcpy(dst, src, n * 4, hipMemcpyDeviceToHost));
            return RBMOE_OK;
        }
        std::vector<uint16_t> tmp(n);
        HIP_TRY(ctx, hipMemcpy(tmp.data(), src, n * 2, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < n; ++i) dst[i] = host_bf16_to_f32(tmp[i]);
        return RBMOE_OK;
    };
    int rc = RBMOE_OK;
    // the hidden rows lie Fw apart; the columns past F are the zeros of the rounded width
    std::vector<float> wide;
    if (L->last_front && hidden && R > 0) {
        // the hidden rows lie per expert over all the call's rows: pick the routed ones, in permuted order
        const int T = L->last_T;
        std::vector<float> all((size_t)E * T * Fw);
        std::vector<int> offs(E + 1), ptok(R);
        rc = fetch(all.data(), L->last.hall, all.size());
        if (rc != RBMOE_OK) return rc;
        HIP_TRY(ctx, hipMemcpy(offs.data(), L->last.offsets, (size_t)(E + 1) * 4, hipMemcpyDeviceToHost));
        HIP_TRY(ctx, hipMemcpy(ptok.data(), L->last.perm_token, (size_t)R * 4, hipMemcpyDeviceToHost));
        for (int e = 0; e < E; ++e)
            for (int pos = offs[e]; pos < offs[e + 1]; ++pos)
                std::memcpy(hidden + (size_t)pos * F, all.data() + ((size_t)e * T + ptok[pos]) * Fw, (size_t)F * 4);
    } else if (hidden && F != Fw) {
        wide.resize((size_t)R * Fw);
        rc = fetch(wide.data(), L->last.h, wide.size());
        if (rc == RBMOE_OK)
            for (int r = 0; r < R; ++r) std::memcpy(hidden + (size_t)r * F, wide.data() + (size_t)r * Fw, (size_t)F * 4);
    } else {
        rc = fetch(hidden, L->last.h, (size_t)R * F);
    }
    if (rc != RBMOE_OK) return rc;
    if (L->last_by_slot && expert_out && R > 0) {
        const int S = L->last_T * L->cfg.experts_per_token;
        std::vector<float> all((size_t)S * d);
        std::vector<int> slots(R);
        rc = fetch(all.data(), L->last.y, all.size());
        if (rc != RBMOE_OK) return rc;
        HIP_TRY(ctx, hipMemcpy(slots.data(), L->last.perm_slot, (size_t)R * 4, hipMemcpyDeviceToHost));
        for (int pos = 0; pos < R; ++pos) std::memcpy(expert_out + (size_t)pos * d, all.data() + (size_t)slots[pos] * d, (size_t)d * 4);
        return RBMOE_OK;
    }
    if (L->last_parts == 1 || !expert_out || R == 0) return fetch(expert_out, L->last.y, (size_t)R * d);
    std::vector<float> part((size_t)R * d);
    for (int p = 0; p < L->last_parts; ++p) {  // a row is the sum of its parts (f32) in order
        const size_t from = (size_t)p * L->last_T * L->cfg.experts_per_token * d;
        HIP_TRY(ctx, hipMemcpy(part.data(), static_cast<const float*>(L->last.y) + from, part.size() * 4, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < part.size(); ++i) expert_out[i] = p == 0 ? part[i] : expert_out[i] + part[i];
    }
    if (abf)
        for (size_t i = 0; i < part.size(); ++i) expert_out[i] = host_bf16_to_f32(host_f32_to_bf16(expert_out[i]));
    return RBMOE_OK;
}

const char* rbmoe_expert_kernel_name(const rbmoe_layer* L) { return L ? L->kernel_name : "none"; }

int rbmoe_device_alloc(rbmoe_ctx* ctx, size_t bytes, void** out) {
    if (!ctx || !out) return fail(ctx, RBMOE_NULL_POINTER, "ctx or out is NULL");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    HIP_TRY(ctx, hipMalloc(out, bytes ? bytes : 1));
    return RBMOE_OK;
}

int rbmoe_device_free(rbmoe_ctx* ctx, void* ptr) {
    if (!ctx) return fail(nullptr, RBMOE_NULL_POINTER, "ctx is NULL");
    if (ptr) HIP_TRY(ctx, hipFree(ptr));
    return RBMOE_OK;
}

int rbmoe_host_alloc(rbmoe_ctx* ctx, size_t bytes, void** out) {
    if (!ctx || !out) return fail(ctx, RBMOE_NULL_POINTER, "ctx or out is NULL");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    *out = host_block_take(bytes ? bytes : 1);
    if (!*out) return fail(ctx, RBMOE_OUT_OF_MEMORY, "the pool of pinned host memory is exhausted");
    return RBMOE_OK;
}

void rbmoe_host_free(void* ptr) {
    if (ptr) host_block_give(ptr);
}

int rbmoe_copy_to_device(rbmoe_ctx* ctx, void* dst, const void* src, size_t bytes) {
    if (!ctx) return fail(nullptr, RBMOE_NULL_POINTER, "ctx is NULL");
    if (bytes == 0) return RBMOE_OK;
    if (!dst || !src) return fail(ctx, RBMOE_NULL_POINTER, "dst or src is NULL");
    HIP_TRY(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return RBMOE_OK;
}

int rbmoe_copy_to_host(rbmoe_ctx* ctx, void* dst, const void* src, size_t bytes) {
    if (!ctx) return fail(nullptr, RBMOE_NULL_POINTER, "ctx is NULL");
    if (bytes == 0) return RBMOE_OK;
    if (!dst || !src) return fail(ctx, RBMOE_NULL_POINTER, "dst or src is NULL");
    HIP_TRY(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return RBMOE_OK;
}

// Test hook (not part of rbmoe.h): the partial matrices an ordered weight-gradient launch over `tokens` tokens cuts
// out, and how many a buffer sized for `max_tokens` holds.
int rbmoe_internal_weight_grad_slots(int32_t M, int32_t N, int32_t groups, int32_t dense, int32_t tokens,
                                     int32_t rows_per_token, int32_t bf16, int32_t max_tokens, int64_t* needed,
                                     int64_t* held) {
    if (!needed || !held) return RBMOE_NULL_POINTER;
    const size_t one = (size_t)M * N * sizeof(float);
    const int rows = dense ? tokens : tokens * rows_per_token;
    *needed = (int64_t)(weight_grad_partial_bytes(M, N, groups, dense ? rows : -1, rows, bf16 != 0) / one);
    *held = (int64_t)(weight_grad_partial_bytes_upto(M, N, groups, dense != 0, max_tokens, rows_per_token, bf16 != 0) / one);
    return RBMOE_OK;
}

// Test hook (not part of rbmoe.h): bytes of the pinned pool in use and kept.
int rbmoe_internal_host_pool(uint64_t* used, uint64_t* kept) {
    if (!used || !kept) return RBMOE_NULL_POINTER;
    size_t u = 0, k = 0;
    host_pool_sizes(&u, &k);
    *used = u;
    *kept = k;
    return RBMOE_OK;
}

// Test hook (not part of rbmoe.h), runs without a GPU: the expert widths that the kernels of a layer see.  out[0]: routed,
// [1]: shared, [2]: 1 mfma_bf16_*, 2 mfma_f32, 0 generic; training != 0: after
// rbmoe_layer_enable_training, RBMOE_UNSUPPORTED where that refuses the widths.
int rbmoe_internal_widths(const rbmoe_config* cfg, int32_t training, int32_t* out) {
    if (!cfg || !out) return RBMOE_NULL_POINTER;
    rbmoe_layer L;
    L.cfg = *cfg;
    L.Fs = cfg->shared_d_ff > 0 ? cfg->shared_d_ff : cfg->d_ff;
    L.max_T = cfg->max_tokens;
    L.max_S = cfg->max_tokens * cfg->experts_per_token;
    choose_kernel_sets(&L);
    if (training && *training_widths_problem(&L)) {
        L.tight = true;
        choose_kernel_sets(&L);
        if (*training_widths_problem(&L)) return RBMOE_UNSUPPORTED;
    }
    out[0] = L.Fw;
    out[1] = L.Fsw;
    out[2] = L.use_stream ? 1 : L.use_f32_mc ? 2 : 0;
    return RBMOE_OK;
}

// The plan of a large-batch call on aligned rows (none of the addresses is read).
static void plan_of_aligned_rows(int32_t d, int32_t E, int32_t k, int32_t T, int32_t bf16, int32_t norm, int32_t quantized, int32_t exact,
                                 RouterPlan* out) {
    RouterArgs a{};
    a.T = T; a.d = d; a.E = E; a.k = k;
    a.allow_fused = true;
    a.exact = exact != 0;
    a.x = reinterpret_cast<void*>((uintptr_t)1 << 20);
    a.wr = static_cast<const float*>(a.x);
    if (quantized) {
        a.wq = static_cast<const int8_t*>(a.x);
        a.wscale = a.wr;
    }
    if (norm) a.norm_w = a.wr;
    a.arrive = reinterpret_cast<int*>((uintptr_t)1 << 20);
    *out = plan_router(a, bf16 != 0);
}

// Test hook (not part of rbmoe.h), runs without a GPU: how a large-batch call on rows at address `x` (never read) is routed.
// out[0]: tokens of a router block as the dispatch counts them, [1]: whether the norm takes a launch of its own, [2]: whether
// the router's launch takes the plan with the arguments it gets, [3]: tokens of a block when the stage is replayed, [4]: whether
// the sums are taken on the matrix cores (`exact`: RouterArgs::exact; a quantized router's values always are).
int rbmoe_internal_router_plan(int32_t d, int32_t E, int32_t k, int32_t T, int32_t bf16, int32_t norm, int32_t quantized, int32_t exact,
                               int32_t fused, uint64_t x, int32_t* out) {
    if (!out) return RBMOE_NULL_POINTER;
    auto at = [](uint64_t address) { return reinterpret_cast<void*>((uintptr_t)address); };
    void* const own = at(1 << 20);  // the layer's own buffers: on an allocation's boundary
    RouterArgs a{};
    a.x = at(x);
    a.wr = static_cast<const float*>(own);
    a.T = T; a.d = d; a.E = E; a.k = k;
    a.allow_fused = fused != 0;
    a.exact = exact != 0;
    if (quantized) {
        a.wq = static_cast<const int8_t*>(own);
        a.wscale = static_cast<const float*>(own);
    }
    if (norm) {
        a.norm_w = static_cast<const float*>(own);
        a.xn_out = own;
    }
    bool apart = false;
    const RouterPlan p = plan_router_behind_norm(a, own, bf16 != 0, &apart);
    out[0] = p.block_tokens;
    out[1] = apart ? 1 : 0;
    out[2] = router_takes(a, p, bf16 != 0) ? 1 : 0;
    out[4] = p.row_exact ? 1 : 0;
    if (a.norm_w) {
        a.x = own;
        a.norm_w = nullptr;
        a.xn_out = nullptr;
    }
    out[3] = plan_router(a, bf16 != 0).block_tokens;
    return RBMOE_OK;
}

// Test hook (not part of rbmoe.h), runs without a GPU: experts of a routing workgroup of a large-batch call on aligned rows, 0
// where a block's experts are not shared out.
int rbmoe_internal_router_slice(int32_t d, int32_t E, int32_t k, int32_t T, int32_t bf16, int32_t norm, int32_t quantized, int32_t exact) {
    RouterPlan p;
    plan_of_aligned_rows(d, E, k, T, bf16, norm, quantized, exact, &p);
    return p.row_slice;
}

// Test hook (not part of rbmoe.h), runs without a GPU: the launch that keeps rows in LDS in such a call.  out[0]: router rows that lie
// there together, 0 where another launch takes the call, [1]: tokens of its blocks, [2]: bytes of LDS of a workgroup.
void rbmoe_internal_router_rows(int32_t d, int32_t E, int32_t k, int32_t T, int32_t bf16, int32_t norm, int32_t quantized, int32_t exact,
                                int32_t* out) {
    RouterPlan p;
    plan_of_aligned_rows(d, E, k, T, bf16, norm, quantized, exact, &p);
    out[0] = p.row_experts;
    out[1] = p.row_experts ? p.block_tokens : 0;
    out[2] = p.row_experts ? (int32_t)p.row_lds : 0;
}

// Test hook (not part of rbmoe.h), runs without a GPU: rows of the tiles of a matrix-core call of so many routed rows.
int rbmoe_internal_stream_tile(int32_t rows, int32_t E, int32_t F, int32_t d) { return stream_tile_m(rows, E, F, d); }

// Test hook (not part of rbmoe.h), runs without a GPU: the parts of the down product's reduction in a large-batch call of T rows, with a
// shared expert of width Fs (0: none) in the launch.  f32_rows: of launch_grouped_f32 (weight_dtype any), otherwise of the matrix-core
// kernels over bf16 rows (bf16 or int8 weights).
int rbmoe_internal_parts(int32_t T, int32_t E, int32_t k, int32_t F, int32_t Fs, int32_t d, int32_t f32_rows, int32_t weight_dtype) {
    const WeightKind wk = weight_dtype == RBMOE_F32 ? WeightKind::F32 : weight_dtype == RBMOE_I8 ? WeightKind::I8 : WeightKind::BF16;
    GroupedArgs g{};
    g.N = d;
    g.K = F;
    g.a = g.w = reinterpret_cast<const void*>((uintptr_t)1 << 20);  // (never read)
    g.w_expert_stride = (size_t)d * F;
    g.tile_m = f32_rows ? f32_tile_m(T * k, E) : kStreamTileM;
    g.max_tiles = (T * k) / g.tile_m + E;
    g.likely_tiles = likely_tiles(T * k, E, g.tile_m);
    g.routed_rows = T * k;
    g.groups = E;
    g.dense_rows = -1;
    if (Fs) g.dense2 = {g.a, g.w, nullptr, d, Fs, T, nullptr, nullptr};
    return f32_rows ? f32_parts(g, wk) : stream_parts(g);
}

// Test hook (not part of rbmoe.h): how the last forward's products ran.  out[0]: rows of the tiles, [1]: parts of the down product's
// reduction, [2]: whether a row or two took launch_decode_down_few.
int rbmoe_internal_last_products(const rbmoe_layer* L, int32_t* out) {
    if (!L || !out) return RBMOE_NULL_POINTER;
    out[0] = L->last_tile_m;
    out[1] = L->last_parts;
    out[2] = L->last_few ? 1 : 0;
    return RBMOE_OK;
}

int rbmoe_copy_device(rbmoe_ctx* ctx, void* dst, const void* src, size_t bytes) {
    if (!ctx) return fail(nullptr, RBMOE_NULL_POINTER, "ctx is NULL");
    if (bytes == 0) return RBMOE_OK;
    if (!dst || !src) return fail(ctx, RBMOE_NULL_POINTER, "dst or src is NULL");
    HIP_TRY(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return RBMOE_OK;
}

}  // extern "C"
