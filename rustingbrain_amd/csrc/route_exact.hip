// Norm (optional), logits and everything behind them for a call's bf16 rows in one launch, where the router's weights allow the
// column lanes' sums on the matrix cores (route_exact_body).
#include <atomic>
#include <type_traits>

#include "routing_device.h"

namespace rbmoe {

template <int TB, int NL, bool NORM>
__global__ __launch_bounds__(kRouterThreads, 2) void route_exact_kernel(RouteRowsArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int from = blockIdx.y * a.slice, to = a.slice ? min(a.E, from + a.slice) : a.E;  // (no slice: one row of workgroups)
    if (blockIdx.y != 0) a.xn_out = nullptr;                                               // (the first slice writes the rows)
    ExactLogits<TB, NL> logits(a, lds_raw);
    logits.folded = !route_exact_body<TB, NL, NORM>(a, blockIdx.x, from, to, a.slice == 0, lds_raw);
    if (logits.folded) __syncthreads();
    if (a.slice && !last_slice<TB>(a, from, to, lds_raw)) return;
    router_tail<1, TB>(lds_raw, blockIdx.x, a.valid, a.T, a.E, a.k, RouteOut{a.P, a.lse, a.expert_of, a.gate_of}, a.rank_in_block,
                       a.blockcnt, a.partial, logits);
}

hipError_t launch_route_exact(const RouterArgs& a, const RouterPlan& p, hipStream_t s) {
    RouteRowsArgs r{a.x, a.wr, a.wq, a.wscale, a.bias, a.valid, a.T, a.d, a.E, a.k, p.row_experts, a.P, a.lse, a.expert_of, a.gate_of,
                    a.rank_in_block, a.blockcnt, a.partial, nullptr, a.norm_w, a.norm_eps, a.xn_out, true, p.row_slice, a.arrive,
                    a.exact_now};
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
#define RB_ROUTE_EXACT(TB, NL)                                                                                  \
    (a.norm_w ? go(std::integral_constant<void (*)(RouteRowsArgs), &route_exact_kernel<TB, NL, true>>{})        \
              : go(std::integral_constant<void (*)(RouteRowsArgs), &route_exact_kernel<TB, NL, false>>{}))
    if (a.wq) return p.block_tokens == 8 ? RB_ROUTE_EXACT(8, 32) : p.block_tokens == 16 ? RB_ROUTE_EXACT(16, 32) : RB_ROUTE_EXACT(32, 32);
    return p.block_tokens == 8 ? RB_ROUTE_EXACT(8, 8) : p.block_tokens == 16 ? RB_ROUTE_EXACT(16, 8) : RB_ROUTE_EXACT(32, 8);
#undef RB_ROUTE_EXACT
}

}  // namespace rbmoe
