// Host memory the GPU reaches directly (a bounded pool of pinned blocks), the copies between it, pageable host
// memory and the device, and the conversions that ride on them.
#pragma once

#include <hip/hip_runtime.h>

#include <stddef.h>
#include <stdint.h>

namespace rbmoe {

// ---- pinned blocks ---------------------------------------------------------------------------------------------
// Pinning is slow (a millisecond for a few megabytes) and a copy to pageable memory that has not been touched yet
// runs at 4 GB/s (page faults; warm pages 18, pinned 57), so blocks are kept for the next taker.  Blocks in use and
// blocks kept together never exceed kHostPoolMax; above it host_block_take returns null and the caller uses pageable
// memory.  Blocks are kept while a context lives (host_pool_hold, host_pool_release): the last one to go gives the kept
// blocks back to the system, and those still in use follow when they are given back.  Any thread may call any of these.
constexpr size_t kHostPoolMax = (size_t)1 << 30;
void* host_block_take(size_t bytes);
void host_block_give(void* p);
bool host_block_holds(const void* p, size_t bytes);  // whether [p, p + bytes) lies inside a block in use
void host_pool_hold();
void host_pool_release();
void host_pool_sizes(size_t* used, size_t* kept);  // bytes

// A block for the length of a scope (null when the pool is exhausted).
struct HostBlock {
    void* p = nullptr;
    HostBlock() = default;
    explicit HostBlock(size_t bytes) : p(host_block_take(bytes)) {}
    HostBlock(HostBlock&& o) noexcept : p(o.p) { o.p = nullptr; }
    HostBlock& operator=(HostBlock&& o) noexcept {
        if (this != &o) {
            reset();
            p = o.p;
            o.p = nullptr;
        }
        return *this;
    }
    HostBlock(const HostBlock&) = delete;
    HostBlock& operator=(const HostBlock&) = delete;
    void reset() {
        if (p) host_block_give(p);
        p = nullptr;
    }
    ~HostBlock() { reset(); }
};

// ---- conversions on the host (nearest even; a NaN stays a quiet NaN) ----------------------------------------------
void host_rows_to_bf16(const float* in, uint16_t* out, size_t n);
void host_rows_to_f32(const uint16_t* in, float* out, size_t n);

// ---- copies by kernel: the destination may be a pinned block -------------------------------------------------------
struct CopySegment {
    const void* src;
    void* dst;
    unsigned int words;  // 4-byte words; both ends 4-byte aligned
};
constexpr int kMaxCopySegments = 10;
hipError_t launch_copy_segments(const CopySegment* segments, int n, hipStream_t s);
// dst[i] = f32(src[i]) of bf16 rows; n a multiple of 4, dst 16-byte and src 8-byte aligned
hipError_t launch_widen_rows(const void* src, float* dst, size_t n, hipStream_t s);

}  // namespace rbmoe
