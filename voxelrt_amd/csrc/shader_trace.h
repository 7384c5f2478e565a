// shader_trace.h - the GLSL traversal ("shader method") per lane.
//
// src/VoxelRT/Shaders/VoxelTraversal.glsl differs from the CPU cast that
// traverse.h reproduces: a clipped start (clipRayToAABB, :133-145), a
// sector-of-sectors LOD level (:110-114), the optional ray-cell interaction
// table (:116-121), a +5 ulp bias (:172), a 256-iteration cap, and a coarse
// variant for shadow and bounce rays (rayCastCoarse, :206-243) that accepts
// any solid voxel of a non-empty 4x4x4 cell from its 31st iteration on.  The
// FP contract is the one stated for vrt_cast_shader in vrt.h.
#pragma once

#include <hip/hip_runtime.h>

#include "traverse.h"
#include "vrt_internal.h"
#include "vrt_math.h"

namespace vrt {

__device__ __forceinline__ bool fine_bit(uint64_t m, uint32_t idx) { return (m >> (idx & 63u)) & 1u; }

// findAnyOccupiedPos (:40-52): v moved to the lowest set bit of its cell's mask, low word first.
__device__ __forceinline__ void first_occupied(uint64_t m, int32_t v[3]) {
    uint32_t bit = (uint32_t)m != 0 ? (uint32_t)__builtin_ctz((uint32_t)m)
                                    : 32u + (uint32_t)__builtin_ctz((uint32_t)(m >> 32));
    v[0] = (v[0] & ~3) | (int32_t)(bit & 3u);
    v[1] = (v[1] & ~3) | (int32_t)((bit >> 4) & 3u);
    v[2] = (v[2] & ~3) | (int32_t)((bit >> 2) & 3u);
}

// getStepPos (:92-131).  Returns true when v is solid (or, for a coarse step, when v
// was moved to the first solid voxel of its non-empty 4x4x4 cell); otherwise moves v
// to the far corner, in ray direction, of the largest empty aligned cell.
template <bool LUT>
__device__ __forceinline__ bool shader_step(const ShaderView& sv, int32_t v[3], const float d[3], uint32_t oct,
                                            bool coarse) {
    const WorldView& w = sv.w;
    uint32_t ux = (uint32_t)v[0], uy = (uint32_t)v[1], uz = (uint32_t)v[2];
    uint32_t sx = ux >> 5, sy = uy >> 5, sz = uz >> 5;
    uint32_t si = sx | sz << w.shift_xz | sy << (2 * w.shift_xz);
    uint4 sec = w.sec[si];
    uint64_t m = (uint64_t)sec.x | (uint64_t)sec.y << 32;
    uint32_t idx = __builtin_amdgcn_ubfe(ux, 3, 2) | __builtin_amdgcn_ubfe(uz, 3, 2) << 2 |
                   __builtin_amdgcn_ubfe(uy, 3, 2) << 4;
    int32_t scale = 8;
    if (fine_bit(m, idx)) {
        uint32_t slot = sec.z + (uint32_t)__popcll(m & ((1ull << idx) - 1ull));
        uint32_t cell = __builtin_amdgcn_ubfe(ux, 2, 1) | __builtin_amdgcn_ubfe(uz, 2, 1) << 1 |
                        __builtin_amdgcn_ubfe(uy, 2, 1) << 2;
        m = w.occ[(size_t)slot * 8 + cell];
        idx = (ux & 3u) | (uz & 3u) << 2 | (uy & 3u) << 4;
        scale = 1;
        if (fine_bit(m, idx)) return true;
    } else if (m == 0) {
        uint32_t gmx = (1u << sv.gshift_xz) - 1u, gmy = (1u << sv.gshift_y) - 1u;
        uint32_t g = ((sx >> 2) & gmx) | ((sz >> 2) & gmx) << sv.gshift_xz | ((sy >> 2) & gmy) << (2 * sv.gshift_xz);
        m = sv.groups[g];
        idx = (sx & 3u) | (sz & 3u) << 2 | (sy & 3u) << 4;
        scale = 32;
    }
    if constexpr (LUT) m &= sv.lut[idx + oct * 64];
    int32_t iso;
    if (m == 0) {
        iso = 4;
    } else {
        uint32_t half = idx < 32 ? (uint32_t)m : (uint32_t)(m >> 32);
        iso = ((half >> (idx & 0xAu)) & 0x00330033u) == 0 ? 2 : 1;
    }
    int32_t lod = iso * scale;
    if (coarse && lod < 4) {
        first_occupied(m, v);
        return true;
    }
    uint32_t cm = (uint32_t)lod - 1u;
#pragma unroll
    for (int a = 0; a < 3; a++)
        v[a] = d[a] < 0.0f ? (int32_t)((uint32_t)v[a] & ~cm) : (int32_t)((uint32_t)v[a] | cm);
    return false;
}

// clipRayToAABB (:133-145) against [1 - W, size - W - 1]; inv: 1 / d.
__device__ __forceinline__ void clip_ray(const WorldView& w, const float o[3], const float d[3], const float inv[3],
                                         const int32_t W[3], float out[3]) {
    float size[3] = {(float)w.size_xz, (float)w.size_y, (float)w.size_xz};
    float lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        float bmin = (float)(int32_t)(1u - (uint32_t)W[a]);
        float bmax = (size[a] - (float)W[a]) - 1.0f;
        float t1 = (bmin - o[a]) * inv[a], t2 = (bmax - o[a]) * inv[a];
        lo[a] = fminf(t1, t2);
        hi[a] = fmaxf(t1, t2);
    }
    float tmin = fmaxf(lo[0], fmaxf(lo[1], lo[2]));
    float tmax = fminf(hi[0], fminf(hi[1], hi[2]));
    bool clip = tmin > 0.0f && tmin < tmax;
#pragma unroll
    for (int a = 0; a < 3; a++) out[a] = clip ? fmaf(d[a], tmin, o[a]) : o[a];
}

// Result of one shader-method trace.
struct ShaderHit {
    float t;        // biased tmin at the hit, -1 on a miss
    float cur[3];   // hit position (relative to W)
    int32_t v[3];   // hit voxel (absolute)
    uint32_t code;  // normal code (vrt_hit info bits 8-13)
    uint32_t iters; // loop index at the hit or miss, the cap when exhausted
    uint32_t mat;   // material id, 0 on a miss
};

// The loop of rayCast / rayCastCoarse for any ray.
template <bool COARSE, bool LUT>
__device__ __forceinline__ bool shader_loop(const ShaderView& sv, const float d[3], const float org[3],
                                            const float inv[3], const float ts[3], const int32_t W[3], uint32_t oct,
                                            uint32_t cap, int32_t v[3], float side[3], float cur[3], float& tmin,
                                            uint32_t& it) {
    const WorldView& w = sv.w;
    bool hit = false;
    for (; it < cap; it++) {
#pragma unroll
        for (int a = 0; a < 3; a++)
            side[a] = fmaf((float)(int32_t)((uint32_t)v[a] - (uint32_t)W[a]), inv[a], ts[a]);
        tmin = fminf(fminf(side[0], side[1]), side[2]);
        if (COARSE)
            tmin = tmin + 0.001f;
        else
            tmin = __uint_as_float(__float_as_uint(tmin) + 5u);
#pragma unroll
        for (int a = 0; a < 3; a++) {
            cur[a] = fmaf(tmin, d[a], org[a]);
            v[a] = (int32_t)((uint32_t)W[a] + (uint32_t)floor2i(cur[a]));
        }
        if (!((uint32_t)(v[0] | v[2]) < w.size_xz && (uint32_t)v[1] < w.size_y)) break;
        if (shader_step<LUT>(sv, v, d, oct, COARSE && it > 30)) {
            hit = true;
            break;
        }
    }
    return hit;
}

// The ray-cell table in a block's LDS, entry oct * 64 + (63 - cell): filled by all of its lanes, each
// a pair of entries at a time, before the first trace.
constexpr uint32_t kLutPairs = 256;
template <bool LUT>
__device__ __forceinline__ uint32_t fill_lut(const ShaderView& sv, uint4* lut) {
    if constexpr (LUT) {
        for (uint32_t p = threadIdx.x; p < kLutPairs; p += blockDim.x) {
            const uint4 e = ((const uint4*)sv.lut)[p];
            lut[p ^ 31u] = make_uint4(e.z, e.w, e.x, e.y);
        }
        __syncthreads();
        return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint4*)lut;
    }
    return 0;
}

// The masked mask v[54:55] of the cell with shifts t1 (its bit, from the top) and t2 (its 2x2x2
// group): the ray-cell table's word, read before the mask arrives (VRT_LUT_READ), and as t0 and t1 the
// mask ored and its 2x2x2 group's (VRT_LUT_MASK).
#define VRT_LUT_READ                                       \
    "v_and_b32 %[t0], 63, %[t1]\n\t"                       \
    "v_lshl_add_u32 %[t0], %[t0], 3, %[lut]\n\t"           \
    "ds_read_b64 v[54:55], %[t0]\n\t"
#define VRT_LUT_MASK(lo, hi)                               \
    "v_and_b32 v54, " lo ", v54\n\t"                       \
    "v_and_b32 v55, " hi ", v55\n\t"
#define VRT_LUT_TESTS                                      \
    "v_or_b32 %[t0], v54, v55\n\t"                         \
    "v_lshrrev_b64 v[54:55], %[t2], v[54:55]\n\t"          \
    "v_and_b32 %[t1], 0x330033, v54\n\t"
// VRT_STEP_SECTOR and VRT_STEP_CELL over the mask table with the ray-cell table.  A record's mask is
// of 8- or 32-voxel cells, w = 3 or 5 their log2.
#define VRT_LUT_SECTOR                                     \
    VRT_STEP_RECORD("%[alive]")                            \
    "v_lshlrev_b32 %[t2], 2, %[g2]\n\t"                    \
    "v_lshlrev_b32 %[t1], 4, %[g1]\n\t"                    \
    "s_waitcnt vmcnt(0)\n\t"                               \
    "v_lshrrev_b32 %[t0], v51, %[g0]\n\t"                  \
    "v_lshrrev_b32 %[t2], v51, %[t2]\n\t"                  \
    "v_lshrrev_b32 %[t1], v51, %[t1]\n\t"                  \
    "v_bitop3_b32 %[t0], 12, %[t2], %[t0] bitop3:0xca\n\t" \
    "v_bitop3_b32 %[t1], 48, %[t1], %[t0] bitop3:0x35\n\t" \
    VRT_LUT_READ                                           \
    "v_bitop3_b32 %[t2], %[t1], 42, %[t1] bitop3:0x0c\n\t" \
    "v_lshlrev_b64 v[52:53], %[t1], v[48:49]\n\t"          \
    "v_bfm_b32 %[cm], v51, 0\n\t"                          \
    "v_cmp_gt_i32 vcc, 0, v53\n\t"                         \
    "s_waitcnt lgkmcnt(0)\n\t"                             \
    VRT_LUT_MASK("v48", "v49")                             \
    VRT_LUT_TESTS                                          \
    "v_sub_u32 %[t0], 1, %[t0] clamp\n\t"                  \
    "v_sub_u32 %[t1], 1, %[t1] clamp\n\t"                  \
    "v_lshl_or_b32 %[t0], %[t0], 1, %[t1]\n\t"             \
    "v_lshl_or_b32 %[cm], %[t0], v51, %[cm]\n\t"
#define VRT_LUT_CELL                                       \
    "v_lshrrev_b32 %[t2], 1, %[g2]\n\t"                    \
    VRT_STEP_CELL_LOAD                                     \
    VRT_LUT_READ                                           \
    "s_waitcnt vmcnt(0)\n\t"                               \
    "v_lshlrev_b64 v[56:57], %[t1], v[52:53]\n\t"          \
    "v_cmp_gt_i32 vcc, 0, v57\n\t"                         \
    "s_waitcnt lgkmcnt(0)\n\t"                             \
    VRT_LUT_MASK("v52", "v53")                             \
    "s_or_b64 %[stop], %[stop], vcc\n\t"                   \
    "v_mov_b32 v52, v54\n\t"                               \
    "v_mov_b32 v53, v55\n\t"                               \
    VRT_LUT_TESTS

// shader_loop for quick rays (ray_is_quick of the start org, d and inv): the cast's fast loop
// (traverse.h) with this method's bias, its level above an empty sector (step records' bits 8..9) and
// rayCastCoarse's stop in a non-empty cell from step 31 on.  The largest cell, 128 voxels, lies inside
// the tables.  Positions stay within their border as there where the distances run from a point of the
// world (rayCastCoarse: from the clipped start).  rayCast's run from the origin itself, so that t covers
// the way to the world and both its rounding and the bias of 5 ulps grow with it: past a cell's far plane
// by up to 2^-23 |o| and 5 2^-23 |o| voxels of each axis.  With |o| below 2^24 on every axis that is 12 of
// the border's 32; rays from further away take shader_loop (ray_starts_near).  A step at the sector level takes 37 vector
// instructions (shader_loop's about 70, with no record kept between steps): 2.07 M camera rays over
// the 1024^3 terrain 167 -> 96 us (rayCast), 80 -> 45 us (rayCastCoarse).  slot: the hit voxel's
// brick.  With the ray-cell table (lut: fill_lut's result plus the ray's octant * 512) a step ands
// the mask of its cell with the table's word, read from LDS, and a step at the sector level takes 46:
// 0.92 M camera rays over the same terrain 69 -> 44 us (coarse), 158 -> 99 us (full).  500 k rays
// with no order in a 64^3 world of noise, which loop up to the cap: 305 -> 181 us, 323 -> 215 with
// the table.
template <bool COARSE, bool LUT>
__device__ __forceinline__ bool shader_loop_fast(const ShaderView& sv, uint32_t lut, const float d[3],
                                                 const float org[3], const float inv[3], const float ts[3], const int32_t W[3],
                                                 const int32_t dm[3], uint32_t cap, int32_t v[3], float side[3],
                                                 float cur[3], float& tmin, uint32_t& steps, uint32_t& slot) {
    const WorldView& w = sv.w;
    // the first step leaves the start's voxel, which may lie anywhere
#pragma unroll
    for (int a = 0; a < 3; a++)
        side[a] = fmaf((float)(int32_t)((uint32_t)v[a] - (uint32_t)W[a]), inv[a], ts[a]);
    tmin = fminf(fminf(side[0], side[1]), side[2]);
    tmin = COARSE ? tmin + 0.001f : __uint_as_float(__float_as_uint(tmin) + 5u);
    float bias3[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        cur[a] = fmaf(tmin, d[a], org[a]);
        bias3[a] = 8388608.0f + (float)(W[a] + kStepPad);
    }
    uint32_t g[3], u[3];
    biased_floor(cur, bias3, g);
#pragma unroll
    for (int a = 0; a < 3; a++) u[a] = g[a] - (0x4B000000u + (uint32_t)kStepPad);
    steps = 0;
    if (!((u[0] | u[2]) < w.size_xz && u[1] < w.size_y)) return false;
    const i32x4 rsec = buffer_rsrc(LUT ? sv.masks : w.steps, 16, w.step_n);
    const i32x4 rocc = buffer_rsrc(w.occ - 8, 8, w.occ_n + 8u);
    uint32_t iters = cap, si = ~0u, slot1 = 0, base, it = 0;
    uint32_t cm, t0, t1, t2, mlo, mhi;
    uint64_t save, alive, stop;
#define VRT_SHADER_STEP(bias, sector, cell, coarse)                                                             \
    asm volatile("s_mov_b64 %[save], exec\n\t"                                                                  \
                 "s_branch vrt_look%=\n\t.p2align 6\n"                                                          \
                 "vrt_advance%=:\n\t" VRT_STEP_ADVANCE("%[tm]", bias) VRT_STEP_FLOOR                            \
                 "vrt_look%=:\n\t" sector                                                                       \
                 "s_cbranch_vccz vrt_advance%=\n\t" cell coarse VRT_STEP_STOP                                   \
                 "vrt_done%=:\n\t"                                                                              \
                 "s_mov_b64 exec, %[save]\n\t"                                                                  \
                 "v_mov_b32 %[base], v50\n\t"                                                                   \
                 "v_mov_b32 %[mlo], v52\n\t"                                                                    \
                 "v_mov_b32 %[mhi], v53"                                                                        \
                 : VRT_STEP_OUT(cur, side, g), [tm] "+&v"(tmin), [mlo] "=&v"(mlo), [mhi] "=&v"(mhi)             \
                 : VRT_STEP_IN(org, d, inv, ts, dm, bias3, cap), [lod] "s"(0x60u), [lut] "v"(lut)               \
                 : VRT_STEP_CLOBBERS, "v56", "v57", "memory")
#define VRT_FINE "v_add_u32 %[tm], 5, %[tm]\n\t"
#define VRT_COARSE "v_add_f32 %[tm], 0x3a83126f, %[tm]\n\t"
// any voxel of the cell stops the ray once it > 30 (t0: its mask, ored)
#define VRT_COARSE_STOP                 \
    "v_cmp_ne_u32 vcc, 0, %[t0]\n\t"    \
    "s_cmp_gt_u32 %[it], 30\n\t"        \
    "s_cselect_b64 vcc, vcc, 0\n\t"     \
    "s_or_b64 %[stop], %[stop], vcc\n\t"
#define VRT_SECTOR               \
    VRT_STEP_SECTOR("%[alive]")  \
    "v_lshrrev_b32 %[t0], 3, v51\n\tv_and_or_b32 %[cm], %[t0], %[lod], %[cm]\n\t"
    if constexpr (COARSE && LUT)
        VRT_SHADER_STEP(VRT_COARSE, VRT_LUT_SECTOR, VRT_LUT_CELL, VRT_COARSE_STOP);
    else if constexpr (COARSE)
        VRT_SHADER_STEP(VRT_COARSE, VRT_SECTOR, VRT_STEP_CELL, VRT_COARSE_STOP);
    else if constexpr (LUT)
        VRT_SHADER_STEP(VRT_FINE, VRT_LUT_SECTOR, VRT_LUT_CELL, "");
    else
        VRT_SHADER_STEP(VRT_FINE, VRT_SECTOR, VRT_STEP_CELL, "");
#undef VRT_SECTOR
#undef VRT_COARSE_STOP
#undef VRT_COARSE
#undef VRT_FINE
#undef VRT_SHADER_STEP
    const bool hit = iters < cap && (int32_t)base >= 0;
    steps = iters;
    slot = slot1 - 1u;
#pragma unroll
    for (int a = 0; a < 3; a++) v[a] = (int32_t)(g[a] & 0x7FFFFFu) - kStepPad;
    if (COARSE && hit) {
        const uint64_t m = (uint64_t)mlo | (uint64_t)mhi << 32;
        const uint32_t vi = ((uint32_t)v[0] & 3u) | ((uint32_t)v[2] & 3u) << 2 | ((uint32_t)v[1] & 3u) << 4;
        if (!fine_bit(m, vi)) first_occupied(m, v);
    }
    return hit;
}

// Whether rayCast's distances, taken from o, keep a ray's positions within the border (shader_loop_fast).
// From 2^26 on they do not: nearly parallel rays then miss the border's records.
__device__ __forceinline__ bool ray_starts_near(const float o[3]) {
    return fmaxf(fmaxf(fabsf(o[0]), fabsf(o[1])), fabsf(o[2])) < 16777216.0f;
}

// rayCast (COARSE = false, :162-204) or rayCastCoarse (COARSE = true, :206-243).  lut: fill_lut's result.
template <bool COARSE, bool LUT>
__device__ __forceinline__ bool shader_trace(const ShaderView& sv, uint32_t lut, const float o[3], const float d[3],
                                             const int32_t W[3], uint32_t cap, ShaderHit& out) {
    const WorldView& w = sv.w;
    float start[3], org[3], inv[3], ts[3], side[3] = {0.0f, 0.0f, 0.0f}, cur[3] = {0.0f, 0.0f, 0.0f};
    int32_t v[3], dm[3];
    auto begin = [&] {
        clip_ray(w, o, d, inv, W, start);
#pragma unroll
        for (int a = 0; a < 3; a++) {
            org[a] = COARSE ? start[a] : o[a];
            ts[a] = ((d[a] < 0.0f ? 0.0f : 1.0f) - org[a]) * inv[a];
            v[a] = (int32_t)((uint32_t)W[a] + (uint32_t)floor2i(start[a]));
            dm[a] = d[a] < 0.0f ? 0 : -1;
        }
    };
    float tmin = 0.0f;
    uint32_t it = 0, slot = 0;
    bool hit;
    const uint32_t oct = (d[0] < 0.0f ? 0u : 1u) + (d[1] < 0.0f ? 0u : 2u) + (d[2] < 0.0f ? 0u : 4u);
#pragma unroll
    for (int a = 0; a < 3; a++) inv[a] = reciprocal_in_range(d[a]);
    begin();
    if (origin_is_guarded(W) && masks_in_reach(w) &&
        __all(ray_is_quick(org, d, inv) && (COARSE || ray_starts_near(org)))) {
        hit = shader_loop_fast<COARSE, LUT>(sv, lut + oct * 512u, d, org, inv, ts, W, dm, cap, v, side, cur, tmin, it,
                                            slot);
    } else {
#pragma unroll
        for (int a = 0; a < 3; a++) inv[a] = 1.0f / d[a];
        begin();
        hit = shader_loop<COARSE, LUT>(sv, d, org, inv, ts, W, oct, cap, v, side, cur, tmin, it);
        if (hit) slot = brick_slot_at(w, v);
    }
    // the record is built in locals and stored once, so the result stays in registers
    uint32_t code = 0, mat = 0;
    float t = -1.0f;
    int32_t hv[3] = {0, 0, 0};
    float hc[3] = {0.0f, 0.0f, 0.0f};
    if (hit) {
#pragma unroll
        for (int a = 0; a < 3; a++)
            if (tmin >= side[a]) code |= (d[a] < 0.0f ? 1u : (d[a] > 0.0f ? 3u : 0u)) << (2 * a);
        uint32_t ux = (uint32_t)v[0], uy = (uint32_t)v[1], uz = (uint32_t)v[2];
        mat = w.vox[(size_t)slot * 512 + ((ux & 7u) | (uz & 7u) << 3 | (uy & 7u) << 6)];
        t = tmin;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            hc[a] = cur[a];
            hv[a] = v[a];
        }
    }
    out.iters = it;
    out.t = t;
    out.code = code;
    out.mat = mat;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        out.cur[a] = hc[a];
        out.v[a] = hv[a];
    }
    return hit;
}

}  // namespace vrt
