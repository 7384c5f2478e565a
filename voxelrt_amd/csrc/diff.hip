// diff.hip - differentiable Lambertian render: forward (cast + shade, saving
// the hit voxel and shading weight of every pixel) and backward (scatter-add
// of dL/dpixel x weight into per-voxel RGB albedo gradients).
//
// No reference counterpart (the reference renders, it does not differentiate);
// the shading term is the reference's sun light: direction
// normalize(0.3, 0.9, -0.28), intensity 5 (Shaders/VoxelRender.comp:133-134)
// with a Lambert N.L factor.  The traversal stays discrete and exact (the same
// cast as vrt_cast), so radiance is linear in the albedo and
//   d radiance_pc / d albedo[v][c] = weight_p  if pixel p hit voxel v.
#include <hip/hip_runtime.h>

#include <cstring>

#include <algorithm>
#include <string>

#include "traverse.h"
#include "vrt_cast_impl.h"

namespace vrt {

// Up to kFwdViews views per launch, their cameras passed in the kernel arguments: one
// launch over many small views fills the chip where one launch per view (a 512x512
// view is half a round of resident waves) leaves it draining after every view.
constexpr uint32_t kFwdViews = 16;
struct FwdViews {
    vrt_camera cam[kFwdViews];
    uint32_t block_begin[kFwdViews + 1];  // first block of 64 pixels of each view; [nv] = all blocks
    uint32_t pixel_base[kFwdViews];       // first output pixel of each view
    tile_map tiles[kFwdViews];
    float inv_w[kFwdViews], inv_h[kFwdViews];
    uint32_t nv;
};

__global__ __launch_bounds__(64) void render_fwd_kernel(WorldView w, FwdViews views, uint32_t max_iters,
                                                        float lx, float ly, float lz, float intensity,
                                                        const float* __restrict__ albedo, float* __restrict__ image,
                                                        uint32_t* __restrict__ saved_voxel,
                                                        float* __restrict__ saved_weight) {
    // the wave's view (blocks never straddle views)
    const uint32_t b = blockIdx.x;
    uint32_t k = 0;
    while (k + 1 < views.nv && b >= views.block_begin[k + 1]) k++;
    const vrt_camera& cam = views.cam[k];
    const uint32_t n = cam.width * cam.height;
    const uint32_t li = (b - views.block_begin[k]) * 64u + threadIdx.x;  // pixel within the view
    const bool valid = li < n;
    const uint32_t i = views.pixel_base[k] + li;                          // output pixel
    RayState st;
    int32_t v[3] = {0, 0, 0};
    if (valid) {
        uint32_t px, py;
        tile_pixel(li, views.tiles[k], px, py);
        float d[3];
        camera_ray(cam.forward, cam.right, cam.up, views.inv_w[k], views.inv_h[k], px, py, d);
        ray_setup(st, cam.eye[0], cam.eye[1], cam.eye[2], d[0], d[1], d[2], cam.world_origin[0], cam.world_origin[1],
                  cam.world_origin[2]);
        uint32_t slot = 0;
        bool hit = ray_trace_wave(w, st, max_iters, v, slot);
        float wgt = 0.0f;
        uint32_t gv = 0xFFFFFFFFu;
        if (hit) {
            float t;
            int4 rec;
            ray_hit_record(w, st, v, slot, t, rec);
            float nx = normal_component((uint32_t)rec.w, 0), ny = normal_component((uint32_t)rec.w, 1),
                  nz = normal_component((uint32_t)rec.w, 2);
            float ndl = nx * lx + ny * ly + nz * lz;
            wgt = fmaxf(ndl, 0.0f) * intensity;
            uint32_t ux = (uint32_t)v[0], uy = (uint32_t)v[1], uz = (uint32_t)v[2];
            gv = slot * 512u + ((ux & 7u) | (uz & 7u) << 3 | (uy & 7u) << 6);
        }
        float r = 0.0f, g = 0.0f, b = 0.0f;
        if (gv != 0xFFFFFFFFu) {
            r = albedo[(size_t)gv * 3 + 0] * wgt;
            g = albedo[(size_t)gv * 3 + 1] * wgt;
            b = albedo[(size_t)gv * 3 + 2] * wgt;
        }
        image[(size_t)i * 3 + 0] = r;
        image[(size_t)i * 3 + 1] = g;
        image[(size_t)i * 3 + 2] = b;
        store_past(saved_voxel + i, gv);
        store_past(saved_weight + i, wgt);
    }
}

__device__ __forceinline__ float wave_masked_sum(float x, bool take) {
    float s = take ? x : 0.0f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    return s;
}

// Scatter-add with wave aggregation: lanes that hit the same voxel are summed
// in registers (ballot on the key of the first pending lane, shuffle
// reduction) and one lane issues the atomics; after kRounds unique keys the
// remaining lanes add directly.
__global__ __launch_bounds__(256) void render_bwd_kernel(uint32_t n, const float* __restrict__ grad_image,
                                                         const uint32_t* __restrict__ saved_voxel,
                                                         const float* __restrict__ saved_weight,
                                                         float* __restrict__ grad_albedo) {
    const int kRounds = 4;
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t gv = 0xFFFFFFFFu;
    float gr = 0.0f, gg = 0.0f, gb = 0.0f;
    if (i < n) {
        gv = saved_voxel[i];
        float wgt = saved_weight[i];
        if (gv != 0xFFFFFFFFu && wgt != 0.0f) {
            gr = grad_image[(size_t)i * 3 + 0] * wgt;
            gg = grad_image[(size_t)i * 3 + 1] * wgt;
            gb = grad_image[(size_t)i * 3 + 2] * wgt;
        } else {
            gv = 0xFFFFFFFFu;
        }
    }
    bool pending = gv != 0xFFFFFFFFu;
    const uint32_t lane = __lane_id();
    for (int round = 0; round < kRounds; round++) {
        uint64_t todo = __ballot(pending);
        if (todo == 0) break;
        uint32_t leader = (uint32_t)__ffsll((unsigned long long)todo) - 1u;
        uint32_t key = __shfl(gv, (int)leader, 64);
        bool mine = pending && gv == key;
        float sr = wave_masked_sum(gr, mine), sg = wave_masked_sum(gg, mine), sb = wave_masked_sum(gb, mine);
        if (lane == leader) {
            atomicAdd(&grad_albedo[(size_t)key * 3 + 0], sr);
            atomicAdd(&grad_albedo[(size_t)key * 3 + 1], sg);
            atomicAdd(&grad_albedo[(size_t)key * 3 + 2], sb);
        }
        if (mine) pending = false;
    }
    if (pending) {
        atomicAdd(&grad_albedo[(size_t)gv * 3 + 0], gr);
        atomicAdd(&grad_albedo[(size_t)gv * 3 + 1], gg);
        atomicAdd(&grad_albedo[(size_t)gv * 3 + 2], gb);
    }
}

// ---------------------------------------------------------------- brick-bucketed backward

// Hit pixels are bucketed by brick slot (a counting sort: per-slot counts with wave-aggregated integer
// atomics, an allocation of the slots' lists, a placement pass), then a workgroup per touched slot
// sums its pixels' contributions in LDS and writes the slot's 512 x 3 gradient entries: no global
// float atomics.  The other entries are zeros, and they are most of it: 16 views of 512 x 512 over the
// 512^3 terrain touch 8.9 k of its 97 k slots (1.7 M pixels, 195 per touched slot).  So the gradient is
// filled with zeros first, at the rate of a fill, and the touched slots are written a second time.
// Measured there (598 MB), in us: fill 77, counts 27, allocation 5, placement 24, sums 19, against 197
// for six launches the last of which wrote each slot's zeros or sums by a wave.  Sharing a launch
// between the fill and the counts or the placement gained nothing (they wait for each other's memory),
// nor did filling after the placement (counts and placement 8 faster, sums 5 slower, a launch more).
constexpr uint32_t kScanBlock = 1024;   // slots per block of the allocation

// Zeros in `vecs` float4s from `out` and the `tail` floats after them, and in `n` words of p.  A float4
// per thread, so that neighbouring blocks fill neighbouring 4 KB: 598 MB in 77.5-82 us, 7.3-7.7 TB/s
// (filled alone again and again 6.9, blocks of 16 and 64 KB 6.1 and 5.1, grids that stride over the
// gradient 4.4-6.1).  first: the launch's first block, as
// gradients past 68 GB need more lanes than a launch has.
__global__ __launch_bounds__(256) void bwd_fill_kernel(float4* __restrict__ out, uint64_t vecs, uint32_t tail,
                                                       uint32_t* __restrict__ p, uint32_t n, uint64_t first) {
    const uint64_t v = (first + blockIdx.x) * 256 + threadIdx.x;
    if (v < vecs)
        out[v] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    else if (v - vecs < tail)
        ((float*)(out + vecs))[v - vecs] = 0.0f;
    else if (v - vecs - tail < n)
        p[v - vecs - tail] = 0u;
}

// Pass 1: the rank of each contributing pixel among the pixels of its slot; counts[slot] ends
// as the slot's pixel count.  Lanes of a wave with the same slot are matched by ballot (eight
// rounds, each for the first pending lane's slot; a lane left over stands for itself), the block's
// slots meet in an LDS table, and each slot in it takes its room with one global atomic.  The
// atomics are performed past the XCDs' L2s and serialize on a slot that fills much of an image: one per
// wave and slot took 33 us for the 16 views and 12.7 for three of 375x281, one per block 26.8 and 7.9
// (blocks of 512 and 1024 pixels 27-30 and 6.2-10).
constexpr uint32_t kCountThreads = 256;
constexpr uint32_t kCountTable = 2 * kCountThreads;  // never more than half full
__global__ __launch_bounds__(kCountThreads) void bwd_count_kernel(uint32_t n, const uint32_t* __restrict__ saved_voxel,
                                                                  const float* __restrict__ saved_weight,
                                                                  uint32_t* __restrict__ counts,
                                                                  uint32_t* __restrict__ rank) {
    __shared__ uint32_t keys[kCountTable], cnt[kCountTable];
    const uint32_t t = threadIdx.x, lane = __lane_id();
    const uint32_t i = blockIdx.x * kCountThreads + t;
    const uint32_t gv = i < n ? saved_voxel[i] : 0xFFFFFFFFu;
    const float weight = i < n ? saved_weight[i] : 0.0f;
#pragma unroll
    for (uint32_t k = t; k < kCountTable; k += kCountThreads) {
        keys[k] = 0xFFFFFFFFu;
        cnt[k] = 0u;
    }
    __syncthreads();
    const bool in = gv != 0xFFFFFFFFu && weight != 0.0f;
    const uint32_t slot = gv >> 9;  // below 2^23
    bool pending = in;
    uint32_t leader = lane;
    uint64_t same = 1ull << lane;
#pragma unroll 1
    for (int k = 0; k < 8; k++) {
        const uint64_t todo = __ballot(pending);
        if (todo == 0) break;  // wave-uniform
        const uint32_t first = (uint32_t)__builtin_ctzll(todo);
        const uint32_t key = __builtin_amdgcn_readlane(slot, first);
        const bool mine = pending && slot == key;
        const uint64_t m = __ballot(mine);
        if (mine) {
            leader = first;
            same = m;
            pending = false;
        }
    }
    // the leaders find their slot's entry: at most 256 of 512 are taken, so a free one ends the search
    uint32_t h = 0, base = 0;
    if (in && leader == lane) {
        h = (slot * 2654435761u) >> (32 - __builtin_ctz(kCountTable));
        for (;;) {
            const uint32_t k = atomicCAS(&keys[h], 0xFFFFFFFFu, slot);
            if (k == 0xFFFFFFFFu || k == slot) break;
            h = (h + 1) & (kCountTable - 1u);
        }
        base = atomicAdd(&cnt[h], (uint32_t)__popcll(same));
    }
    __syncthreads();
    uint32_t from[2];
#pragma unroll
    for (uint32_t p = 0; p < 2; p++) {
        const uint32_t k = keys[t + p * kCountThreads];
        from[p] = k != 0xFFFFFFFFu ? atomicAdd(&counts[k], cnt[t + p * kCountThreads]) : 0u;
    }
#pragma unroll
    for (uint32_t p = 0; p < 2; p++) cnt[t + p * kCountThreads] = from[p];
    __syncthreads();
    if (in && leader == lane) base += cnt[h];
    base = __shfl(base, (int)leader, 64);
    const uint32_t before =
        __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
    if (i < n) rank[i] = in ? base + before : 0xFFFFFFFFu;
}

// Pass 2: the slots' lists and the list of the touched slots.  A block scans kScanBlock counts
// (256 threads x 4) and takes its room in both lists with one atomic each, so the lists' order
// varies between runs, as the ranks do.
__global__ __launch_bounds__(256) void bwd_alloc_kernel(uint32_t ns, const uint32_t* __restrict__ counts,
                                                        uint32_t* __restrict__ cursor, uint32_t* __restrict__ offsets,
                                                        uint4* __restrict__ touched) {
    __shared__ uint64_t wave_total[4];
    __shared__ uint32_t start[2];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t base = blockIdx.x * kScanBlock + t * 4;
    uint32_t c[4];
    uint64_t sum = 0;  // pixels, and touched slots in the high half (a block holds at most 2^10)
#pragma unroll
    for (int k = 0; k < 4; k++) {
        c[k] = base + k < ns ? counts[base + k] : 0u;
        sum += (uint64_t)c[k] | (uint64_t)(c[k] != 0) << 32;
    }
    uint64_t incl = sum;
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        uint64_t y = __shfl_up((unsigned long long)incl, off, 64);
        if (lane >= off) incl += y;
    }
    if (lane == 63) wave_total[wave] = incl;
    __syncthreads();
    uint64_t run = incl - sum;
    for (uint32_t w = 0; w < wave; w++) run += wave_total[w];
    if (t == 255) {
        const uint64_t total = run + sum;
        start[0] = (uint32_t)total ? atomicAdd(&cursor[0], (uint32_t)total) : 0u;
        start[1] = (uint32_t)total ? atomicAdd(&cursor[1], (uint32_t)(total >> 32)) : 0u;
    }
    __syncthreads();
    uint32_t px = start[0] + (uint32_t)run, ts = start[1] + (uint32_t)(run >> 32);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (c[k] == 0) continue;
        offsets[base + k] = px;
        touched[ts++] = make_uint4(base + k, px, c[k], 0u);
        px += c[k];
    }
}

// Pass 3: each contributing pixel's contribution, grad_image * weight, and voxel as one 16-byte entry at
// its slot's offset plus its rank.  (With the pixel's index there instead, 11 us and not 24, the next
// pass gathers the pixels' data and takes 39 us and not 19: a slot's pixels are runs of 8 or so in an
// 8x8 tile, and most of each line fetched for them belongs to other slots.)
__global__ __launch_bounds__(256) void bwd_place_kernel(uint32_t n, const float* __restrict__ grad_image,
                                                        const uint32_t* __restrict__ saved_voxel,
                                                        const float* __restrict__ saved_weight,
                                                        const uint32_t* __restrict__ rank,
                                                        const uint32_t* __restrict__ offsets,
                                                        float4* __restrict__ list) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t r = rank[i];
    if (r == 0xFFFFFFFFu) return;
    const uint32_t gv = saved_voxel[i];
    const float w = saved_weight[i];
    const float x = grad_image[(size_t)i * 3 + 0] * w, y = grad_image[(size_t)i * 3 + 1] * w,
                z = grad_image[(size_t)i * 3 + 2] * w;
    list[offsets[gv >> 9] + r] = make_float4(x, y, z, __uint_as_float(gv & 511u));
}

// Pass 4: one workgroup per touched slot, striding over them (their number is on the device).  The
// slot's entries are added into 512 x 3 LDS accumulators, then the workgroup writes the slot's rows
// [slot * 512, min(nvox, slot * 512 + 512)) of the gradient.  The accumulators are doubles: an LDS
// atomic add of 64 floats takes this part 194 cycles, of doubles 18-22 (the adds alone held this pass
// at 50 us with floats), and the sums are rounded once.  Bound by latency: the next slot's place is
// loaded ahead, and a thread has kReducePixels entries in flight.  Each XCD (workgroup b runs on XCD
// b % 8) takes an eighth of the slots in a piece.
constexpr uint32_t kReduceThreads = 128;
constexpr uint32_t kReduceBlocks = 3072;  // 12 per CU: 12 KB of LDS each, of 160
constexpr uint32_t kReducePixels = 2;

__global__ __launch_bounds__(kReduceThreads) void bwd_reduce_kernel(uint64_t nvox,
                                                                    const uint32_t* __restrict__ cursor,
                                                                    const uint4* __restrict__ touched,
                                                                    const float4* __restrict__ list,
                                                                    float* __restrict__ grad_albedo) {
    __shared__ __align__(16) double acc[512 * 3];
    const uint32_t t = threadIdx.x, ntouched = cursor[1];
    const uint32_t per = (ntouched + 7) / 8, first = (blockIdx.x & 7u) * per, end = min(first + per, ntouched);
    uint32_t s = first + (blockIdx.x >> 3);
    if (s >= end) return;
    uint4 next = touched[s];
    while (s < end) {
        const uint32_t slot = next.x, begin = next.y, cnt = next.z;
        s += gridDim.x >> 3;
        if (s < end) next = touched[s];  // ahead of its use
        for (uint32_t k = t; k < 768; k += kReduceThreads) ((double2*)acc)[k] = make_double2(0.0, 0.0);
        __syncthreads();
        for (uint32_t j0 = 0; j0 < cnt; j0 += kReduceThreads * kReducePixels) {
            float4 e[kReducePixels];
#pragma unroll
            for (uint32_t q = 0; q < kReducePixels; q++)
                e[q] = list[begin + min(j0 + q * kReduceThreads + t, cnt - 1u)];
#pragma unroll
            for (uint32_t q = 0; q < kReducePixels; q++) {
                if (j0 + q * kReduceThreads + t >= cnt) continue;
                double* a = acc + __float_as_uint(e[q].w) * 3;
                atomicAdd(a + 0, (double)e[q].x);
                atomicAdd(a + 1, (double)e[q].y);
                atomicAdd(a + 2, (double)e[q].z);
            }
        }
        __syncthreads();
        const uint64_t row0 = (uint64_t)slot * 512;
        const uint32_t rows = (uint32_t)min<uint64_t>(512, nvox - row0);
        float* out = grad_albedo + row0 * 3;
        if (rows == 512) {
            for (uint32_t k = t; k < 384; k += kReduceThreads)
                ((float4*)out)[k] = make_float4((float)acc[k * 4], (float)acc[k * 4 + 1], (float)acc[k * 4 + 2],
                                                (float)acc[k * 4 + 3]);
        } else {
            for (uint32_t k = t; k < rows * 3; k += kReduceThreads) out[k] = (float)acc[k];
        }
        __syncthreads();
    }
}

// Sparse gradient: entry p is (voxel id, grad_image[p] * weight[p]), or (0, 0) for a pixel that
// contributes nothing (a miss or zero weight); duplicates are summed by whoever coalesces.
__global__ __launch_bounds__(256) void bwd_sparse_kernel(uint32_t n, const float* __restrict__ grad_image,
                                                         const uint32_t* __restrict__ saved_voxel,
                                                         const float* __restrict__ saved_weight,
                                                         int64_t* __restrict__ index, float* __restrict__ values) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t gv = saved_voxel[i];
    float w = saved_weight[i];
    bool take = gv != 0xFFFFFFFFu && w != 0.0f;
    index[i] = take ? (int64_t)gv : 0;
    values[(size_t)i * 3 + 0] = take ? grad_image[(size_t)i * 3 + 0] * w : 0.0f;
    values[(size_t)i * 3 + 1] = take ? grad_image[(size_t)i * 3 + 1] * w : 0.0f;
    values[(size_t)i * 3 + 2] = take ? grad_image[(size_t)i * 3 + 2] * w : 0.0f;
}

// Workspace of the brick-bucketed backward: two cursors and the counts (cleared together), offsets
// (one u32 per slot each), the touched slots (slot, first entry, count), ranks (one u32 per pixel)
// and the entries (16 bytes per pixel), each part 256-byte aligned.
struct BwdWorkspace {
    uint32_t *cursor, *counts, *offsets, *rank;
    uint4* touched;
    float4* list;
};
constexpr uint32_t kCursorWords = 64;  // before the counts

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

static size_t bwd_workspace_bytes(uint32_t npixels, uint64_t nslots) {
    return kCursorWords * 4 + 2 * align256(nslots * 4) + std::min<uint64_t>(nslots, npixels) * 16 + 256 +
           align256((size_t)npixels * 4) + align256((size_t)npixels * 16);
}

static BwdWorkspace carve_bwd(void* base, uint32_t npixels, uint64_t nslots) {
    char* p = (char*)base;
    BwdWorkspace ws;
    ws.cursor = (uint32_t*)p; p += kCursorWords * 4;
    ws.counts = (uint32_t*)p; p += align256(nslots * 4);
    ws.offsets = (uint32_t*)p; p += align256(nslots * 4);
    ws.touched = (uint4*)p; p += align256(std::min<uint64_t>(nslots, npixels) * 16);
    ws.rank = (uint32_t*)p; p += align256((size_t)npixels * 4);
    ws.list = (float4*)p;
    return ws;
}

}  // namespace vrt

using namespace vrt;

extern "C" {

int vrt_render_fwd(const vrt_world* world, const vrt_camera* cameras, uint32_t nviews, uint32_t max_iters,
                   const float light_dir[3], float intensity, const float* albedo, float* image,
                   uint32_t* saved_voxel, float* saved_weight, void* stream) {
    return guarded([&]() -> int {
        if (!world || (nviews && !cameras) || !light_dir)
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_fwd: null argument");
        if (int rcw = check_world(world, "vrt_render_fwd"); rcw != VRT_OK) return rcw;
        if (max_iters == 0 || max_iters > 65535) return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_fwd: max_iters must be 1..65535");
        if ((uint64_t)world->slot_cap * 512 >= 0xFFFFFFFFull)
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_fwd: world too large for 32-bit voxel ids");
        hipStream_t s = (hipStream_t)stream;
        WorldView w = world->view();
        uint64_t total = 0;
        for (uint32_t k = 0; k < nviews; k++) {
            const vrt_camera& c = cameras[k];
            if (!c.width || !c.height || !c.tile_w || !c.tile_h || c.width % c.tile_w || c.height % c.tile_h)
                return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_fwd: camera size must be a multiple of its tile");
            total += (uint64_t)c.width * c.height;
        }
        // each launch's 64-lane blocks (at most one partial block per view) and every
        // output pixel index must fit in 32 bits
        if (total > 0xFFFFF000ull) return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_fwd: more than 2^32 - 4096 pixels");
        if (total && (!albedo || !image || !saved_voxel || !saved_weight))
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_fwd: null argument");
        uint32_t base = 0;
        for (uint32_t k0 = 0; k0 < nviews; k0 += kFwdViews) {
            FwdViews v{};
            v.nv = std::min(kFwdViews, nviews - k0);
            uint64_t blocks = 0;
            for (uint32_t k = 0; k < v.nv; k++) {
                const vrt_camera& c = cameras[k0 + k];
                v.cam[k] = c;
                v.block_begin[k] = (uint32_t)blocks;
                v.pixel_base[k] = base;
                v.tiles[k] = make_tile_map(c.width, c.tile_w, c.tile_h);
                v.inv_w[k] = 1.0f / (float)c.width;
                v.inv_h[k] = 1.0f / (float)c.height;
                uint32_t n = c.width * c.height;
                blocks += ((uint64_t)n + 63) / 64;
                base += n;
            }
            v.block_begin[v.nv] = (uint32_t)blocks;
            render_fwd_kernel<<<(uint32_t)blocks, 64, 0, s>>>(w, v, max_iters, light_dir[0], light_dir[1], light_dir[2],
                                                               intensity, albedo, image, saved_voxel, saved_weight);
            VRT_HIP(hipGetLastError());
        }
        return VRT_OK;
    });
}

int vrt_render_bwd(const vrt_world* world, uint32_t npixels, const float* grad_image, const uint32_t* saved_voxel,
                   const float* saved_weight, float* grad_albedo, void* stream) {
    return guarded([&]() -> int {
        if (!world || (npixels && (!grad_image || !saved_voxel || !saved_weight || !grad_albedo)))
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd: null argument");
        if (int rcw = check_world(world, "vrt_render_bwd"); rcw != VRT_OK) return rcw;
        if (npixels == 0) return VRT_OK;
        if (npixels > 0xFFFFFF00u) return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd: more than 2^32 - 256 pixels");
        render_bwd_kernel<<<(npixels + 255) / 256, 256, 0, (hipStream_t)stream>>>(npixels, grad_image, saved_voxel,
                                                                                  saved_weight, grad_albedo);
        VRT_HIP(hipGetLastError());
        return VRT_OK;
    });
}

size_t vrt_render_bwd_workspace_bytes(uint32_t npixels, uint64_t nvox) {
    return bwd_workspace_bytes(npixels, (nvox + 511) / 512);
}

int vrt_render_bwd_bricks(const vrt_world* world, uint32_t npixels, const float* grad_image,
                          const uint32_t* saved_voxel, const float* saved_weight, uint64_t nvox, float* grad_albedo,
                          void* workspace, size_t workspace_bytes, void* stream) {
    return guarded([&]() -> int {
        if (!world) return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_bricks: null world");
        if (int rcw = check_world(world, "vrt_render_bwd_bricks"); rcw != VRT_OK) return rcw;
        if (npixels > 0xFFFFFF00u) return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_bricks: more than 2^32 - 256 pixels");
        // every saved id is below slot_high_water * 512 (the world is unchanged since the forward pass)
        const uint64_t need = (uint64_t)world->arena.high_water() * 512;
        if (nvox < need)
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_bricks: nvox " + std::to_string(nvox) +
                                                      " < slot_high_water * 512 = " + std::to_string(need));
        const uint64_t nslots = (nvox + 511) / 512;
        if (nslots > kMaxSlots) return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_bricks: nvox above 2^37");
        if (nvox == 0) return VRT_OK;
        if (!grad_albedo || !workspace || (npixels && (!grad_image || !saved_voxel || !saved_weight)))
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_bricks: null argument");
        if (workspace_bytes < bwd_workspace_bytes(npixels, nslots))
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_bricks: workspace smaller than "
                                                  "vrt_render_bwd_workspace_bytes(npixels, nvox)");
        if (((uintptr_t)grad_albedo & 15) != 0 || ((uintptr_t)workspace & 255) != 0)
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_bricks: grad_albedo must be 16-byte and the "
                                                  "workspace 256-byte aligned");
        hipStream_t s = (hipStream_t)stream;
        BwdWorkspace ws = carve_bwd(workspace, npixels, nslots);
        const uint32_t ns = (uint32_t)nslots, nblk = (uint32_t)((nslots + kScanBlock - 1) / kScanBlock);
        // kernels, not memsets (graph-safe); the counts and cursors are cleared with the gradient
        const uint64_t vecs = nvox * 3 / 4;
        const uint32_t tail = (uint32_t)(nvox * 3 % 4), words = npixels ? ns + kCursorWords : 0u;
        const uint64_t fill = (vecs + tail + words + 255) / 256;
        for (uint64_t first = 0; first < fill;) {
            const uint32_t blocks = launch_blocks(fill - first, 256);
            bwd_fill_kernel<<<blocks, 256, 0, s>>>((float4*)grad_albedo, vecs, tail, ws.cursor, words, first);
            // every pass indexes by what the passes before it wrote: none after one that failed
            VRT_HIP(hipGetLastError());
            first += blocks;
        }
        if (npixels) {
            bwd_count_kernel<<<(npixels + kCountThreads - 1) / kCountThreads, kCountThreads, 0, s>>>(
                npixels, saved_voxel, saved_weight, ws.counts, ws.rank);
            VRT_HIP(hipGetLastError());
            bwd_alloc_kernel<<<nblk, 256, 0, s>>>(ns, ws.counts, ws.cursor, ws.offsets, ws.touched);
            VRT_HIP(hipGetLastError());
            bwd_place_kernel<<<(npixels + 255) / 256, 256, 0, s>>>(npixels, grad_image, saved_voxel, saved_weight, ws.rank,
                                                                   ws.offsets, ws.list);
            VRT_HIP(hipGetLastError());
            const uint32_t blocks = std::min({ns, npixels, kReduceBlocks});
            bwd_reduce_kernel<<<(blocks + 7) / 8 * 8, kReduceThreads, 0, s>>>(nvox, ws.cursor, ws.touched, ws.list,
                                                                             grad_albedo);
            VRT_HIP(hipGetLastError());
        }
        return VRT_OK;
    });
}

int vrt_render_bwd_sparse(const vrt_world* world, uint32_t npixels, const float* grad_image,
                          const uint32_t* saved_voxel, const float* saved_weight, int64_t* index, float* values,
                          void* stream) {
    return guarded([&]() -> int {
        if (!world) return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_sparse: null world");
        if (int rcw = check_world(world, "vrt_render_bwd_sparse"); rcw != VRT_OK) return rcw;
        if (npixels == 0) return VRT_OK;
        if (!grad_image || !saved_voxel || !saved_weight || !index || !values)
            return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_sparse: null argument");
        if (npixels > 0xFFFFFF00u) return fail(VRT_ERR_INVALID_ARGUMENT, "vrt_render_bwd_sparse: more than 2^32 - 256 pixels");
        bwd_sparse_kernel<<<(npixels + 255) / 256, 256, 0, (hipStream_t)stream>>>(npixels, grad_image, saved_voxel,
                                                                                  saved_weight, index, values);
        VRT_HIP(hipGetLastError());
        return VRT_OK;
    });
}

}  // extern "C\"
