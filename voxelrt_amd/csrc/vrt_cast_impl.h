// vrt_cast_impl.h - kernel-side ray/hit views shared by the cast, bounce,
// batched and differentiable translation units (not part of the ABI).
#pragma once

#include <hip/hip_runtime.h>

#include "vrt_internal.h"

namespace vrt {

// Stores of results and loads of rays that the launch does not touch again (non-temporal): kept, their
// lines push the world's tables and cells out of an XCD's 4 MiB L2.  Stores: 24 cameras with 8 ray sets
// 480 -> 447 us, 1920x1080 primary and bounce rays 152.6 -> 146.9, a 640x360 preview with the full record
// 19.0 -> 18.2, 2 M rays without order 376 -> 370, frames and the shader method 1%.  The compact schedule's
// ray loads: 370 -> 352.  Rays that the launch before wrote are still in a cache: with such loads 1920x1080
// primary rays took 69.3 us and not 63.5, so the grid's are plain; so are the differentiable image's
// stores, 12 bytes a lane (388 -> 399).
template <class T>
__device__ __forceinline__ void store_past(T* p, T v) {
    if constexpr (sizeof(T) == 16) {
        typedef uint32_t words __attribute__((ext_vector_type(4)));
        __builtin_nontemporal_store(__builtin_bit_cast(words, v), (words*)p);
    } else {
        __builtin_nontemporal_store(v, p);
    }
}
__device__ __forceinline__ float load_past(const float* p) { return __builtin_nontemporal_load(p); }

struct RaysIn {
    const float* __restrict__ ox;
    const float* __restrict__ oy;
    const float* __restrict__ oz;
    const float* __restrict__ dx;
    const float* __restrict__ dy;
    const float* __restrict__ dz;
    int32_t W[3];
    uint32_t n;                        // capacity
    const uint32_t* __restrict__ count;  // optional device ray count (<= n)
};

// Rays to trace: the device count when given, clamped to the capacity.
__device__ __forceinline__ uint32_t ray_count(const RaysIn& r) {
    return r.count ? min(*r.count, r.n) : r.n;
}

struct HitsOut {
    float* __restrict__ t;
    int4* __restrict__ rec;
    float* __restrict__ pos_x;  // all three null when positions are not requested
    float* __restrict__ pos_y;
    float* __restrict__ pos_z;
    float* __restrict__ uv_u;   // both null when texture coordinates are not requested
    float* __restrict__ uv_v;
    uint32_t* __restrict__ material_data;  // null when not requested
    const uint64_t* __restrict__ palette;  // the world's palette (material_data)
};

// ---------------------------------------------------------------- work queues
constexpr uint32_t kQueues = 8;
constexpr uint32_t kQueueStride = 64;  // u32 per counter (256 bytes)

struct ChunkQueue {
    uint32_t* ctr;          // kQueues counters, kQueueStride apart, zero at launch
    uint32_t nchunks;       // total chunks
    uint32_t waves_per_q;   // waves with a static first chunk in each part
};

__device__ __forceinline__ uint32_t part_begin(uint32_t q, uint32_t nchunks) {
    return (uint32_t)(((uint64_t)nchunks * q) / kQueues);
}

// Next chunk for this wave, or ~0u when every part is drained.  Wave-uniform.
__device__ __forceinline__ uint32_t claim_chunk(const ChunkQueue& cq, uint32_t home, uint32_t& probe) {
    while (probe < kQueues) {
        uint32_t q = (home + probe) % kQueues;
        uint32_t b = part_begin(q, cq.nchunks), e = part_begin(q + 1, cq.nchunks);
        uint32_t k = 0;
        if (__lane_id() == 0) k = atomicAdd(cq.ctr + q * kQueueStride, 1u);
        k = __shfl(k, 0, 64);
        uint32_t c = b + cq.waves_per_q + k;
        if (c < e) return c;
        probe++;
    }
    return ~0u;
}


// Validates the ABI structs and converts them to kernel views; with extras = false the
// optional uv and material_data outputs are rejected (entry points that do not fill them).
int check_rays_hits(const vrt_rays* rays, const vrt_hits* hits, RaysIn& r, HitsOut& h, bool extras = false);
// Launches a cast with the given options on stream s.
int launch_cast(const vrt_world* world, const RaysIn& r, const HitsOut& h, uint32_t max_iters,
                const vrt_cast_opts& o, hipStream_t s);
// Compute units of device `dev` and, when queue is not null, the queue counters of persistent
// launches on stream s of that device (kQueues counters, kQueueStride apart).
int device_info(int dev, int* cus, uint32_t** queue, hipStream_t s);

}  // namespace vrt
