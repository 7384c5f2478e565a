// device_checks.hip - what tests/test_gpu_device_facts.py and test_bwd_large.py call beside the ABI: kernels
// for facts about this part that the traversal's loops rest on, through the functions that the loops use
// (traverse.h), a world's slot arena, and the split of large launches.
#include <hip/hip_runtime.h>

#include "traverse.h"

namespace {

using vrt::i32x4;

// out[k] = record index[k] of the structured buffer, as the loops load them (ray_trace_fast).
__global__ __launch_bounds__(64) void load8_kernel(const void* table, uint32_t records,
                                                   const uint32_t* __restrict__ index, uint32_t n,
                                                   uint64_t* __restrict__ out) {
    const uint32_t k = blockIdx.x * 64 + threadIdx.x;
    if (k >= n) return;
    const i32x4 rsrc = vrt::buffer_rsrc(table, 8, records);
    uint64_t v;
    asm volatile("buffer_load_dwordx2 %0, %1, %2, 0 idxen\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(v) : "v"(index[k]), "s"(rsrc) : "memory");
    out[k] = v;
}
__global__ __launch_bounds__(64) void load16_kernel(const void* table, uint32_t records,
                                                    const uint32_t* __restrict__ index, uint32_t n,
                                                    i32x4* __restrict__ out) {
    const uint32_t k = blockIdx.x * 64 + threadIdx.x;
    if (k >= n) return;
    const i32x4 rsrc = vrt::buffer_rsrc(table, 16, records);
    i32x4 v;
    asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 idxen\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(v) : "v"(index[k]), "s"(rsrc) : "memory");
    out[k] = v;
}

// Thread m: the numbers of mantissa m, of both signs and exponents lo to hi, whose reciprocal differs.
__global__ __launch_bounds__(256) void reciprocal_kernel(int lo, int hi, uint32_t* __restrict__ differ) {
    const uint32_t m = blockIdx.x * 256 + threadIdx.x;
    uint32_t bad = 0;
    for (int e = lo; e <= hi; e++)
        for (uint32_t s = 0; s < 2; s++) {
            const float x = __uint_as_float(s << 31 | (uint32_t)(e + 127) << 23 | m);
            bad += __float_as_uint(vrt::reciprocal_in_range(x)) != __float_as_uint(1.0f / x);
        }
    if (bad) atomicAdd(differ, bad);
}

}  // namespace

extern "C" {

// stride 8 or 16; index and out hold n entries on the device, the table `records` records.
int check_structured_loads(const void* table, uint32_t stride, uint32_t records, const uint32_t* index, uint32_t n,
                           void* out, void* stream) {
    if (stride != 8 && stride != 16) return (int)hipErrorInvalidValue;
    if (stride == 8)
        load8_kernel<<<(n + 63) / 64, 64, 0, (hipStream_t)stream>>>(table, records, index, n, (uint64_t*)out);
    else
        load16_kernel<<<(n + 63) / 64, 64, 0, (hipStream_t)stream>>>(table, records, index, n, (i32x4*)out);
    return (int)hipGetLastError();
}

// Takes the first n free slots of a world without bricks, which then puts its bricks after them.
int check_take_slots(vrt_world* world, uint32_t n) {
    uint32_t base = 0;
    return world->arena.realloc(base, 0, n) && base == 0 ? 0 : 1;
}

// Blocks of each launch of a kernel of `blocks` blocks in all; their number.
uint32_t check_launches(uint64_t blocks, uint32_t threads, uint32_t* each, uint32_t max) {
    uint32_t n = 0;
    for (uint64_t first = 0; first < blocks && n < max; first += each[n++])
        each[n] = vrt::launch_blocks(blocks - first, threads);
    return n;
}

// -126 <= lo <= hi <= 127; differ: one count on the device, added to.
int check_reciprocals(int lo, int hi, uint32_t* differ, void* stream) {
    reciprocal_kernel<<<1u << 15, 256, 0, (hipStream_t)stream>>>(lo, hi, differ);
    return (int)hipGetLastError();
}

}  // extern "C"
