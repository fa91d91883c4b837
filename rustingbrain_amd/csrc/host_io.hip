#include "host_io.h"

#include <cstring>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "rbmoe_kernels.h"

namespace rbmoe {

namespace {

struct HostPool {
    std::mutex mutex;
    std::map<uintptr_t, size_t> used;              // blocks in use, by address
    std::map<size_t, std::vector<void*>> kept;     // free blocks, by size
    size_t used_bytes = 0, kept_bytes = 0;
    int holders = 0;                               // contexts that live
};

// (never destroyed: blocks may be given back while the process ends)
HostPool& pool() {
    static HostPool* const p = new HostPool();
    return *p;
}

// Blocks come in sizes of eight steps an octave, so that a kept block fits requests of about its own size.
size_t block_size(size_t bytes) {
    if (bytes <= 4096) return 4096;
    size_t top = 4096;
    while (top * 2 <= bytes) top *= 2;
    const size_t step = top / 8 < 4096 ? 4096 : top / 8;
    return (bytes + step - 1) / step * step;
}

void drop_kept(HostPool& p, size_t room) {  // frees kept blocks, largest first, until `room` more bytes fit
    while (p.used_bytes + p.kept_bytes + room > kHostPoolMax && !p.kept.empty()) {
        auto it = std::prev(p.kept.end());
        (void)hipHostFree(it->second.back());
        p.kept_bytes -= it->first;
        it->second.pop_back();
        if (it->second.empty()) p.kept.erase(it);
    }
}

}  // namespace

void* host_block_take(size_t bytes) {
    const size_t size = block_size(bytes);
    if (size > kHostPoolMax) return nullptr;
    HostPool& p = pool();
    std::lock_guard<std::mutex> lock(p.mutex);
    void* block = nullptr;
    auto it = p.kept.find(size);
    if (it != p.kept.end()) {
        block = it->second.back();  // the one given back last
        it->second.pop_back();
        if (it->second.empty()) p.kept.erase(it);
        p.kept_bytes -= size;
    } else {
        if (p.used_bytes + size > kHostPoolMax) return nullptr;
        drop_kept(p, size);
        if (hipHostMalloc(&block, size, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        void* seen_by_gpu = nullptr;
        if (hipHostGetDevicePointer(&seen_by_gpu, block, 0) != hipSuccess || seen_by_gpu != block) {
            (void)hipGetLastError();  // the copy kernels take host addresses as they are
            (void)hipHostFree(block);
            return nullptr;
        }
    }
    p.used.emplace((uintptr_t)block, size);
    p.used_bytes += size;
    return block;
}

void host_block_give(void* block) {
    HostPool& p = pool();
    std::lock_guard<std::mutex> lock(p.mutex);
    auto it = p.used.find((uintptr_t)block);
    if (it == p.used.end()) return;
    const size_t size = it->second;
    p.used.erase(it);
    p.used_bytes -= size;
    if (p.holders == 0) {  // nobody is left to take it again
        (void)hipHostFree(block);
        return;
    }
    p.kept[size].push_back(block);
    p.kept_bytes += size;
}

bool host_block_holds(const void* ptr, size_t bytes) {
    HostPool& p = pool();
    std::lock_guard<std::mutex> lock(p.mutex);
    auto it = p.used.upper_bound((uintptr_t)ptr);
    if (it == p.used.begin()) return false;
    --it;
    return (uintptr_t)ptr + bytes <= it->first + it->second;
}

void host_pool_hold() {
    HostPool& p = pool();
    std::lock_guard<std::mutex> lock(p.mutex);
    ++p.holders;
}

void host_pool_sizes(size_t* used, size_t* kept) {
    HostPool& p = pool();
    std::lock_guard<std::mutex> lock(p.mutex);
    *used = p.used_bytes;
    *kept = p.kept_bytes;
}

void host_pool_release() {
    HostPool& p = pool();
    std::lock_guard<std::mutex> lock(p.mutex);
    if (--p.holders > 0) return;
    for (auto& k : p.kept)
        for (void* b : k.second) (void)hipHostFree(b);
    p.kept.clear();
    p.kept_bytes = 0;
}

// ---------------------------------------------------------------------------
// Conversions on the host: memory-bound once the loops are eight lanes wide.
// ---------------------------------------------------------------------------
#if defined(__HIP_DEVICE_COMPILE__)
#define RB_HOST_SIMD
#else
#define RB_HOST_SIMD __attribute__((target_clones("avx2", "default")))
#endif

RB_HOST_SIMD void host_rows_to_bf16(const float* in, uint16_t* out, size_t n) {
    for (size_t i = 0; i < n; ++i) {
        uint32_t b;
        std::memcpy(&b, in + i, 4);
        const uint32_t rounded = (b + 0x7fffu + ((b >> 16) & 1u)) >> 16;
        const uint32_t quiet = (b >> 16) | 0x0040u;
        out[i] = (uint16_t)((b & 0x7fffffffu) > 0x7f800000u ? quiet : rounded);
    }
}

RB_HOST_SIMD void host_rows_to_f32(const uint16_t* in, float* out, size_t n) {
    for (size_t i = 0; i < n; ++i) {
        const uint32_t b = (uint32_t)in[i] << 16;
        std::memcpy(out + i, &b, 4);
    }
}

// ---------------------------------------------------------------------------
// Copies by kernel
// ---------------------------------------------------------------------------
struct CopySegments {
    CopySegment s[kMaxCopySegments];
};

// Several small arrays in one launch, blockIdx.y = array: as separate DMA copies they cost 10 to 15 us each, whatever
// their size.
__global__ __launch_bounds__(256) void copy_segments_kernel(CopySegments a) {
    const CopySegment g = a.s[blockIdx.y];
    const uint32_t* const src = static_cast<const uint32_t*>(g.src);
    uint32_t* const dst = static_cast<uint32_t*>(g.dst);
    const unsigned int stride = gridDim.x * 256u;
    for (unsigned int i = blockIdx.x * 256u + threadIdx.x; i < g.words; i += stride) dst[i] = src[i];
}

hipError_t launch_copy_segments(const CopySegment* segments, int n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (n > kMaxCopySegments) return hipErrorInvalidValue;
    CopySegments a{};
    unsigned int widest = 1;
    for (int i = 0; i < n; ++i) {
        a.s[i] = segments[i];
        if (segments[i].words > widest) widest = segments[i].words;
    }
    const unsigned int blocks = (widest + 1023) / 1024;
    hipLaunchKernelGGL(copy_segments_kernel, dim3(blocks < 64 ? blocks : 64, n), dim3(256), 0, s, a);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void widen_rows_kernel(const bf16_t* __restrict__ src, float* __restrict__ dst, size_t n4) {
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += stride) {
        const uint2 v = reinterpret_cast<const uint2*>(src)[i];
        reinterpret_cast<float4*>(dst)[i] = make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                                                        __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u));
    }
}

hipError_t launch_widen_rows(const void* src, float* dst, size_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    if (n % 4) return hipErrorInvalidValue;
    const size_t n4 = n / 4, blocks = (n4 + 255) / 256;
    hipLaunchKernelGGL(widen_rows_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0, s,
                       static_cast<const bf16_t*>(src), dst, n4);
    return hipGetLastError();
}

}  // namespace rbmoe
