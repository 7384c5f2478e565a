// traverse.h - the per-ray brickmap DDA on the device.
//
// One lane owns one ray.  The arithmetic is the reference CPU cast
// (src/VoxelRT/CpuRenderer.cpp:135-224) per lane: FP32, IEEE 1/d, explicit
// fmaf for sideDist and the next position, x86 min and floor2i semantics,
// +0.001 bias, 2-level LOD from the 64-bit masks (brick level 8/16/32 voxels,
// voxel level 1/2/4).  Storage is the popcount-compacted GPU layout
// (GpuRenderer.cpp:27-33, VoxelMap.glsl:45-64) with the sector's mask and
// base slot packed in one 16-byte record, so a lookup is one load.
//
// Two instantiations of the step compute identical traversals:
//   EXACT = true   floor2i with x86 cvtps2dq semantics (NaN / out of range ->
//                  INT_MIN) and x86 minps (a < b ? a : b) in the loop;
//   EXACT = false  plain floor + convert and v_min3_f32, valid for "tame" rays
//                  (finite 1/d and tStart, |o| < 2^20, 0.25 <= |d|^2 <= 4):
//                  their positions stay far inside int32 range for any
//                  iteration cap (a step moves at most 32*sqrt(3)/|d| + 0.001
//                  along d, i.e. < 56 voxels, and 65535 * 56 + 2^20 < 2^31),
//                  and their side distances are never NaN, so floor2i never
//                  takes its INT_MIN branch and the two minimums agree up to
//                  the sign of a zero, which cannot change tmin + 0.001.
// The reported t is recomputed with the exact x86 minimum in both cases.
//
// The two are steps of the exact loop and of the persistent schedules.  Every other kernel goes
// through ray_trace_wave, whose fast loop (below) makes the same traversal with fewer
// instructions, at any world origin W.
#pragma once

#include <hip/hip_runtime.h>

#include "vrt_internal.h"
#include "vrt_math.h"

namespace vrt {

struct RayState {
    float o[3], d[3], inv[3], ts[3], side[3], cur[3];
    int32_t W[3];
    int32_t dm[3];  // all ones where d >= 0: the cell corner to step to is the far one
    uint32_t iters, descents;
    // the sector record of the last lookup and its index (~0u before the first): a step
    // whose position is still in that sector reuses it instead of loading it again
    uint32_t rec_si;
    uint32_t rec[4];
};

enum StepResult : int { STEP_CONTINUE = 0, STEP_HIT = 1, STEP_MISS = 2 };

// 1 / x by V_RCP_F32 and one Newton step on its residual (Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990): the correctly rounded quotient for every
// x with 2^-100 <= |x| < 2^101 (compared with 1.0f / x over all of them on this part), in 3
// instructions instead of the 10 of a division.  Zeros, infinities and NaN give no such value.
__device__ __forceinline__ float reciprocal_in_range(float x) {
    const float q = __builtin_amdgcn_rcpf(x);
    return fmaf(fmaf(-x, q, 1.0f), q, q);
}

// 1 / d and tStart by IEEE division, for any direction.
__device__ __forceinline__ void ray_exact_inverse(RayState& r) {
#pragma unroll
    for (int a = 0; a < 3; a++) {
        r.inv[a] = 1.0f / r.d[a];
        r.ts[a] = ((r.d[a] < 0.0f ? 0.0f : 1.0f) - r.o[a]) * r.inv[a];
    }
}

// A ray at its origin, for ray_trace_wave: 1 / d is right for the directions of quick rays
// (ray_is_quick) only, and ray_trace_wave divides for the others.
__device__ __forceinline__ void ray_setup(RayState& r, float ox, float oy, float oz, float dx, float dy, float dz,
                                          int32_t wx, int32_t wy, int32_t wz) {
    r.o[0] = ox; r.o[1] = oy; r.o[2] = oz;
    r.d[0] = dx; r.d[1] = dy; r.d[2] = dz;
    r.W[0] = wx; r.W[1] = wy; r.W[2] = wz;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        r.inv[a] = reciprocal_in_range(r.d[a]);
        r.ts[a] = ((r.d[a] < 0.0f ? 0.0f : 1.0f) - r.o[a]) * r.inv[a];
        r.side[a] = 0.0f;
        r.cur[a] = r.o[a];
        r.dm[a] = r.d[a] < 0.0f ? 0 : -1;
        // a per-lane word, so the cell alignment below is one bitfield insert per axis
        asm volatile("" : "+v"(r.dm[a]));
    }
    r.iters = 0;
    r.descents = 0;
    // no index reaches ~0u (worlds hold at most 2^27 sectors), and an index past the
    // records reads 0, like this initial record
    r.rec_si = ~0u;
    r.rec[0] = r.rec[1] = r.rec[2] = r.rec[3] = 0;
}

// The same for the loops that step with ray_advance.
__device__ __forceinline__ void ray_setup_exact(RayState& r, float ox, float oy, float oz, float dx, float dy, float dz,
                                                int32_t wx, int32_t wy, int32_t wz) {
    ray_setup(r, ox, oy, oz, dx, dy, dz, wx, wy, wz);
    ray_exact_inverse(r);
}

// True when the fast step is exact for this ray (see the file comment).
__device__ __forceinline__ bool ray_is_tame(const RayState& r) {
    bool ok = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        ok = ok && fabsf(r.inv[a]) < INFINITY && fabsf(r.ts[a]) < INFINITY && fabsf(r.o[a]) < 1048576.0f;
    }
    float len2 = r.d[0] * r.d[0] + r.d[1] * r.d[1] + r.d[2] * r.d[2];
    return ok && len2 >= 0.25f && len2 <= 4.0f;
}

// (mask & a) | (~mask & b): V_BFI_B32.
__device__ __forceinline__ uint32_t bitfield_insert(uint32_t mask, uint32_t a, uint32_t b) {
    return (mask & a) | (~mask & b);
}

// Structured buffer load (BUFFER_LOAD_DWORDX4 ... IDXEN): record vindex of the
// resource's array, the byte address index * stride computed by the load itself, and
// 0 for an index at or past the resource's record count (range-checked in hardware).
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
__device__ i32x4 vrt_struct_buffer_load_v4i32(i32x4 rsrc, int32_t vindex, int32_t voffset, int32_t soffset,
                                              int32_t aux) __asm("llvm.amdgcn.struct.buffer.load.v4i32");

// Buffer resource of the sector records: base address, 16-byte stride, one record per
// sector.  Word 3 is the gfx9 untyped-buffer configuration.
__device__ __forceinline__ i32x4 sector_records_rsrc(const WorldView& w) {
    uint64_t a = (uint64_t)w.sec;
    i32x4 r;
    r.x = (int32_t)(uint32_t)a;
    r.y = (int32_t)(((uint32_t)(a >> 32) & 0xFFFFu) | (16u << 16));
    r.z = (int32_t)(1u << (2 * w.shift_xz + w.shift_y));
    r.w = 0x00020000;
    return r;
}

// (a << sh) | b in one V_LSHL_OR_B32.
__device__ __forceinline__ uint32_t lshl_or(uint32_t a, uint32_t sh, uint32_t b) {
    uint32_t r;
    asm("v_lshl_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(sh), "v"(b));
    return r;
}

// (M & a) | (~M & b) in one V_BFI_B32 for a constant field mask M (written out,
// because the compiler splits a constant-mask insert into ANDs once it knows which
// result bits are used).
template <uint32_t M>
__device__ __forceinline__ uint32_t insert_bits(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "i"(M), "v"(a), "v"(b));
    return r;
}

// ~((M & a) | (~M & b)) in one V_BITOP3_B32: the truth table is indexed by
// (M bit) * 4 + (a bit) * 2 + (b bit), so 0x35 is "not (M ? a : b)".
template <uint32_t M>
__device__ __forceinline__ uint32_t insert_bits_not(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0x35" : "=v"(r) : "i"(M), "v"(a), "v"(b));
    return r;
}

// min(x, 1) in one V_MIN_U32 (the compiler would compare and select).
__device__ __forceinline__ uint32_t min_1(uint32_t x) {
    uint32_t r;
    asm("v_min_u32 %0, %1, 1" : "=v"(r) : "v"(x));
    return r;
}

// floor(x) as int32 in one V_CVT_FLR_I32_F32; x finite and |x| < 2^31.
__device__ __forceinline__ int32_t floor_i32_in_range(float x) {
    int32_t f;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(f) : "v"(x));
    return f;
}

// One iteration of RayCast (CpuRenderer.cpp:185-202) with GetStepPos (:135-171).
// On STEP_HIT, v is the hit voxel and *hit_slot its brick slot.
//
// Integer work is arranged for few VALU instructions per iteration:
//   mask bit test: below = m << (63 - bi) moves bit bi to bit 63 and drops the
//     bits above it, so the test is a sign test and popcount(below) counts the
//     bricks at or below bi, i.e. slot + 1 (the occupancy load subtracts the
//     one as a constant offset);
//   index fields: only bits 0..5 of the in-mask indices are meaningful; the
//     64-bit shifts read only those bits (the & 63 costs nothing), and the
//     fields are merged with bitfield inserts;
//   cell mask: cm = 2^s - 1 with s = level + (group empty) + (mask empty), the
//     reference's LOD of +1 / +2 (a 4x4x4 mask that is 0 has every group empty).
//     With ce = 2^(level + 1 + (mask empty)) - 1, the mask of an empty group, this
//     is cm = ce >> min(group bits, 1); the sector record holds ce for its mask;
//   alignment: (v & ~cm) | (dm & cm), one bitfield insert per axis.
// Occupancy indices slot * 8 + cell are 32-bit: worlds hold at most 2^28 slots.
template <bool EXACT>
__device__ __forceinline__ bool ray_advance(const WorldView& w, RayState& r, int32_t v[3], bool& hit,
                                            uint32_t* hit_slot) {
    int32_t f[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        f[a] = EXACT ? floor2i(r.cur[a]) : floor_i32_in_range(r.cur[a]);
        v[a] = (int32_t)((uint32_t)r.W[a] + (uint32_t)f[a]);
    }
    // GetInboundMask (:114-117)
    if (!((uint32_t)(v[0] | v[2]) < w.size_xz && (uint32_t)v[1] < w.size_y)) {
        hit = false;
        return false;
    }
    r.iters++;
    // a per-lane count: left to itself the compiler derives it from a wave-uniform loop
    // counter with three copies per step
    asm volatile("" : "+v"(r.iters));
    uint32_t ux = (uint32_t)v[0], uy = (uint32_t)v[1], uz = (uint32_t)v[2];
    uint32_t si = lshl_or(uy >> 5, 2 * w.shift_xz, lshl_or(uz >> 5, w.shift_xz, ux >> 5));
    // one 16-byte load for the whole record: a descent then waits on one load (the
    // occupancy mask) instead of two (a structured buffer load: the hardware scales the
    // index, one instruction fewer than a 64-bit address).  A lane still in the sector of
    // its previous step keeps that record and issues no load: divergent waves (bounce and
    // incoherent rays) then send L1 fewer distinct lines per step, and a wave whose lanes
    // all stay skips the load and its wait.  The compare and the copies out of the kept
    // record cost 5 VALU instructions per step; measured, the coherent primary launch
    // takes them without slowing, incoherent sets cast 9-17% faster.
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    if (si != r.rec_si) {
        const u32x4 ld = (u32x4)vrt_struct_buffer_load_v4i32(sector_records_rsrc(w), (int32_t)si, 0, 0, 0);
        r.rec[0] = ld.x;
        r.rec[1] = ld.y;
        r.rec[2] = ld.z;
        r.rec[3] = ld.w;
        r.rec_si = si;
    }
    u32x4 sec;
    sec.x = r.rec[0];
    sec.y = r.rec[1];
    sec.z = r.rec[2];
    sec.w = r.rec[3];
    uint64_t m = (uint64_t)sec.x | (uint64_t)sec.y << 32;
    // brick within the sector: bits 3..4 of x, z, y at bits 0..1, 2..3, 4..5
    // nbi = ~bi: bits 0..5 give the shift 63 - bi, and ~nbi & 0x2A the 2x2x2 group's shift
    uint32_t nbi = insert_bits_not<0x30u>(uy << 1, insert_bits<0x0Cu>(uz >> 1, ux >> 3));
    uint64_t below = m << (nbi & 63u);
    bool descend = (int32_t)(below >> 32) < 0;
    // the cell mask of a step whose 2x2x2 group is empty: 15 below a sector mask, 31
    // when that mask is 0 (from the record); 1 below a voxel mask, 3 when it is 0
    uint32_t ce = sec.w;
    bool solid = false;
    uint32_t slot1 = 0;
    if (descend) {
        r.descents++;
        slot1 = sec.z + (uint32_t)__popcll(below);
        uint32_t cell = __builtin_amdgcn_ubfe(ux, 2, 1) | __builtin_amdgcn_ubfe(uz, 2, 1) << 1 |
                        __builtin_amdgcn_ubfe(uy, 2, 1) << 2;
        m = w.occ[(size_t)(slot1 * 8u + cell) - 8u];
        // voxel within the brick's 4x4x4 cell: bits 0..1 of x, z, y
        nbi = insert_bits_not<0x30u>(uy << 4, insert_bits<0x0Cu>(uz << 2, ux));
        solid = (int32_t)((m << (nbi & 63u)) >> 32) < 0;
        ce = m == 0 ? 3u : 1u;
    }
    // the hit test after the join: its complement is then a scalar mask operation rather than a
    // second vector compare of the sector mask
    if (solid) {
        *hit_slot = slot1 - 1;
        hit = true;
        return false;
    }
    // the 2x2x2 group holding bi: (half >> (bi & 0xA)) & 0x00330033 on the 32-bit
    // half selected by bit 5 of bi
    uint32_t grp = (uint32_t)(m >> (~nbi & 0x2Au)) & 0x00330033u;
    uint32_t cm = ce >> min_1(grp);
#pragma unroll
    for (int a = 0; a < 3; a++) {
        // d < 0: v & ~cm (near corner); d >= 0: v | cm (far corner); rel = that corner - W
        v[a] = (int32_t)bitfield_insert(~cm, (uint32_t)v[a], (uint32_t)r.dm[a]);
        const int32_t rel = (int32_t)((uint32_t)v[a] - (uint32_t)r.W[a]);
        r.side[a] = fmaf((float)rel, r.inv[a], r.ts[a]);
    }
    float tmin;
    if (EXACT)
        tmin = min_x86(min_x86(r.side[0], r.side[1]), r.side[2]);
    else
        tmin = fminf(fminf(r.side[0], r.side[1]), r.side[2]);
    tmin += 0.001f;
#pragma unroll
    for (int a = 0; a < 3; a++) r.cur[a] = fmaf(tmin, r.d[a], r.o[a]);
    return true;
}

// ray_advance as a result code.
template <bool EXACT>
__device__ __forceinline__ int ray_step(const WorldView& w, RayState& r, int32_t v[3], uint32_t* hit_slot) {
    bool hit;
    if (ray_advance<EXACT>(w, r, v, hit, hit_slot)) return STEP_CONTINUE;
    return hit ? STEP_HIT : STEP_MISS;
}

// Brick slot of voxel v, which lies in an allocated brick (a hit voxel): the
// lookup of a descending step, repeated once after the loop so the loop does
// not carry the slot.
// The record is read by the range-checked structured load: an index past the records
// reads 0 (slot = 0), so no v can make this lookup leave the world's buffers.
__device__ __forceinline__ uint32_t brick_slot_at(const WorldView& w, const int32_t v[3]) {
    uint32_t ux = (uint32_t)v[0], uy = (uint32_t)v[1], uz = (uint32_t)v[2];
    uint32_t si = (ux >> 5) | (uz >> 5) << w.shift_xz | (uy >> 5) << (2 * w.shift_xz);
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 sec = (u32x4)vrt_struct_buffer_load_v4i32(sector_records_rsrc(w), (int32_t)si, 0, 0, 0);
    uint64_t m = (uint64_t)sec.x | (uint64_t)sec.y << 32;
    uint32_t bi = __builtin_amdgcn_ubfe(ux, 3, 2) | __builtin_amdgcn_ubfe(uz, 3, 2) << 2 |
                  __builtin_amdgcn_ubfe(uy, 3, 2) << 4;
    return sec.z + (uint32_t)__popcll(m & ((1ull << bi) - 1ull));
}

// ---------------------------------------------------------------- the fast loop

// The same traversal as ray_advance, arranged for this part's issue rates.  With several waves on a
// SIMD a wave64 instruction issues in 2 cycles when it is one of the simple ones with vector
// operands (f32 add, multiply and fma, and / or / xor, right shifts, adds, V_BITOP3_B32), and in 4
// when it is another (conversions, compares, minima, bitfield inserts and extracts, left and 64-bit
// shifts, V_OR3 and the like) or reads a scalar register.  Both kinds measured with 8 waves per
// SIMD: 2.1-2.5 and 4.1-4.3 cycles.  A step that stays at the sector level takes 35 vector
// instructions, 7 of them of the slow kind, and 9 scalar ones and branches (ray_advance: 47, 27
// and 23):
//   position     g = position + bias rounded down, bias = 2^23 + W + kStepPad: the bits of g are
//                2^23's with the padded voxel coordinate in the mantissa, so one addition in the
//                round-down mode replaces a floor, a conversion and an addition (three axes with
//                both mode writes: 9.6 cycles, against 21.9), and after the cell alignment
//                g - bias is the corner relative to W as a float, exactly, with no conversion;
//   bounds       none: the tables have a border (vrt_internal.h) whose records stop the ray;
//   cell mask    the record holds it per 2x2x2 group (step_record);
//   exits        one branch, taken when some lane is in an allocated brick or outside.
// 1920x1080 frames of the 1024^3 terrain (primary and bounce rays): 234 -> 193 us with forward
// blocks; 24 cameras and 8 ray sets in one launch: 579 -> 501 us.  The loop is no longer bound by
// vector issue: a wave waits for its loads (a 16-byte load of 64 lanes takes an L1 17 cycles
// however few lanes are active or lines are read) and the launch for its longest waves.
// It is written out because the compiler's loop spends 8 more scalar instructions and a branch per
// step on lane masks for the exits (one wave alone: 183 against 162 ns per step; ray_advance's
// loop 219).  Waits for the loads are inside the same statement.  Its start is at a 64-byte line: 0.5%
// on the frames, 2% in the shader method.
//
// Quick and guarded rays.  The border is one sector wide, so no position may leave the world by 32
// voxels or more before its lookup.  A position is o + t d with t the least of the three computed
// side distances, plus 0.001.  With u = 2^-24, a side distance is off by at most 2u (|o| + 1) / |d|
// plus a relative 2u (1 / d, the difference, the product and the fma round once each, and the
// error of 1 / d is common to both terms).  t exceeds no side distance, so on each axis the
// position passes the cell's far plane by at most 2u (|o| + 1) + 0.002.  It can fall behind when
// the axis that gives the minimum is far off: by 2u (|o| + 1) |1 / d| |d'| on another axis, less than
// 30.1 voxels where (|o| + 1) |1 / d| times the length of d is at most 30 2^23.  A ray of which this
// holds on every axis, with 0.25 <= |d|^2 <= 4, is quick (its 1 / d and tStart are then finite).  On an
// axis where it does not (a component nudged from zero, say), the axis must never give the minimum:
// the distance to its next voxel plane, over |d| and less the error, exceeds every t in the world.
// Either way the ray is guarded.  Rays that are neither take ray_advance's step, with their wave.
constexpr float kQuickSquare = 251658240.0f * 251658240.0f;  // (30 2^23)^2
__device__ __forceinline__ bool ray_is_quick(const float o[3], const float d[3], const float inv[3]) {
    // the sum bounds each axis, and a NaN on any axis fails the test
    float x = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; a++) x += (fabsf(o[a]) + 1.0f) * fabsf(inv[a]);
    const float len2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    return x * x * len2 <= kQuickSquare && fabsf(len2 - 2.125f) <= 1.875f;
}

__device__ __forceinline__ bool ray_is_guarded(const WorldView& w, const RayState& r) {
    // t of any step in the world: the longest axis of d is at least 0.28
    const float t_max = 8.0f * (float)max(w.size_xz, w.size_y);
    const float len2 = r.d[0] * r.d[0] + r.d[1] * r.d[1] + r.d[2] * r.d[2];
    bool ok = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float inv = fabsf(r.inv[a]), x = (fabsf(r.o[a]) + 1.0f) * inv;
        const float fr = r.o[a] - floorf(r.o[a]);
        const float dist = r.d[a] < 0.0f ? fr : 1.0f - fr;
        ok = ok && (x * x * len2 <= kQuickSquare || dist * inv > t_max + x * 2.384185791015625e-7f);
    }
    return ok;
}

// The biased coordinates need |W| well below 2^23.
__device__ __forceinline__ bool origin_is_guarded(const int32_t W[3]) {
    bool ok = true;
#pragma unroll
    for (int a = 0; a < 3; a++) ok = ok && (uint32_t)(W[a] + (1 << 20)) <= (1u << 21);
    return ok;
}

// Whether a structured load reaches every mask.  This part cuts its index times its stride to 32 bits
// (index 2^29 of a table of 8-byte records reads record 0), and the base is a slot early (ray_trace_fast).
// Worlds that hold memory for more bricks than 2^26 - 1 take ray_advance's step, with 64-bit addresses.
__device__ __forceinline__ bool masks_in_reach(const WorldView& w) { return w.occ_n <= (1u << 29) - 8u; }

// cur + bias per axis, rounded down.
__device__ __forceinline__ void biased_floor(const float cur[3], const float bias[3], uint32_t g[3]) {
    asm("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\t"
        "v_add_f32 %0, %3, %6\n\t"
        "v_add_f32 %1, %4, %7\n\t"
        "v_add_f32 %2, %5, %8\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0"
        : "=&v"(g[0]), "=&v"(g[1]), "=&v"(g[2])
        : "v"(cur[0]), "v"(cur[1]), "v"(cur[2]), "v"(bias[0]), "v"(bias[1]), "v"(bias[2]));
}

__device__ __forceinline__ i32x4 buffer_rsrc(const void* base, uint32_t stride, uint32_t records) {
    uint64_t a = (uint64_t)base;
    i32x4 r;
    r.x = (int32_t)(uint32_t)a;
    r.y = (int32_t)(((uint32_t)(a >> 32) & 0xFFFFu) | (stride << 16));
    r.z = (int32_t)records;
    r.w = 0x00020000;
    return r;
}

// What the record's index is too large by with the border's first sector and the coordinates' exponent
// bits left in: 2^23's bits >> 5, of which the products take the low 24.  Negated.  (Taking the bits out of
// each coordinate is three bitfield extracts of 4 cycles for three shifts of 2 and an addition: 0.6% on
// the frames.)
__device__ __forceinline__ uint32_t step_bias(const WorldView& w) {
    constexpr uint32_t e = 0x4B000000u >> 5, e24 = e & 0xFFFFFFu;
    return 0u - (e + kStepFirst + (e24 + kStepFirst) * (w.step_z + w.step_y));
}

// The parts of the fast loop (operands: ray_trace_fast).  Fixed registers: v[48:51] the kept
// sector record, v[52:55] temporaries, v[56:57] the kept group word.
// The side distances of the cell mask cm and the next position; bias: what is added to the least
// of them (in register tmin).
#define VRT_STEP_ADVANCE(tmin, bias)                           \
    "v_bitop3_b32 %[t0], %[cm], %[m0], %[g0] bitop3:0xca\n\t"  \
    "v_bitop3_b32 %[t1], %[cm], %[m1], %[g1] bitop3:0xca\n\t"  \
    "v_bitop3_b32 %[t2], %[cm], %[m2], %[g2] bitop3:0xca\n\t"  \
    "v_sub_f32 %[t0], %[t0], %[b0]\n\t"                        \
    "v_sub_f32 %[t1], %[t1], %[b1]\n\t"                        \
    "v_sub_f32 %[t2], %[t2], %[b2]\n\t"                        \
    "v_fma_f32 %[s0], %[t0], %[i0], %[ts0]\n\t"                \
    "v_fma_f32 %[s1], %[t1], %[i1], %[ts1]\n\t"                \
    "v_fma_f32 %[s2], %[t2], %[i2], %[ts2]\n\t"                \
    "s_add_u32 %[it], %[it], 1\n\t"                            \
    "v_min3_f32 " tmin ", %[s0], %[s1], %[s2]\n\t"             \
    "s_cmp_ge_u32 %[it], %[max]\n\t"                           \
    bias                                                       \
    "v_fma_f32 %[c0], " tmin ", %[d0], %[o0]\n\t"              \
    "v_fma_f32 %[c1], " tmin ", %[d1], %[o1]\n\t"              \
    "v_fma_f32 %[c2], " tmin ", %[d2], %[o2]\n\t"              \
    "s_cbranch_scc1 vrt_done%=\n\t"
#define VRT_STEP_BIAS "v_add_f32 %[t0], 0x3a83126f, %[t0]\n\t" /* + 0.001 */
// The biased voxel coordinates: position + bias, rounded down.
#define VRT_STEP_FLOOR                                         \
    "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\t"       \
    "v_add_f32 %[g0], %[c0], %[b0]\n\t"                        \
    "v_add_f32 %[g1], %[c1], %[b1]\n\t"                        \
    "v_add_f32 %[g2], %[c2], %[b2]\n\t"                        \
    "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\t"
// The group word, loaded by the lanes that have entered another group, and the sector's bit of
// it: lanes of an empty sector get its cell mask, and the rest go on with exec holding them
// (alive holds all).
#define VRT_STEP_GROUP                                         \
    "v_bfe_u32 %[t0], %[g0], 7, 13\n\t"                        \
    "v_bfe_u32 %[t1], %[g1], 7, 13\n\t"                        \
    "v_bfe_u32 %[t2], %[g2], 7, 13\n\t"                        \
    "v_mad_u32_u24 %[t2], %[t2], %[gz], %[t0]\n\t"             \
    "v_mad_u32_u24 %[t1], %[t1], %[gy], %[t2]\n\t"             \
    "v_cmp_ne_u32 vcc, %[t1], %[gi]\n\t"                       \
    "s_and_saveexec_b64 %[alive], vcc\n\t"                     \
    "s_cbranch_execz vrt_group%=\n\t"                          \
    "buffer_load_dwordx2 v[56:57], %[t1], %[rgrp], 0 idxen\n\t" \
    "v_mov_b32 %[gi], %[t1]\n"                                 \
    "vrt_group%=:\n\t"                                         \
    "s_mov_b64 exec, %[alive]\n\t"                             \
    "v_lshrrev_b32 %[t2], 3, %[g2]\n\t"                        \
    "v_lshrrev_b32 %[t0], 5, %[g0]\n\t"                        \
    "v_lshrrev_b32 %[t1], 1, %[g1]\n\t"                        \
    "v_bitop3_b32 %[t0], 12, %[t2], %[t0] bitop3:0xca\n\t"     \
    "v_bitop3_b32 %[t0], 48, %[t1], %[t0] bitop3:0x35\n\t"     \
    "v_mov_b32 %[cm], 31\n\t"                                  \
    "s_waitcnt vmcnt(0)\n\t"                                   \
    "v_lshlrev_b64 v[52:53], %[t0], v[56:57]\n\t"              \
    "v_cmp_gt_i32 vcc, 0, v53\n\t"                             \
    "s_cbranch_vccz vrt_advance%=\n\t"                         \
    "s_mov_b64 exec, vcc\n\t"
// The sector record, loaded by the lanes that have entered another sector (lanes: what to save
// exec in).
#define VRT_STEP_RECORD(lanes)                                 \
    "v_lshrrev_b32 %[t0], 5, %[g0]\n\t"                        \
    "v_lshrrev_b32 %[t1], 5, %[g1]\n\t"                        \
    "v_lshrrev_b32 %[t2], 5, %[g2]\n\t"                        \
    "v_mad_u32_u24 %[t2], %[t2], %[sz], %[t0]\n\t"             \
    "v_mad_u32_u24 %[t1], %[t1], %[sy], %[t2]\n\t"             \
    "v_add_u32 %[t1], %[t1], %[sk]\n\t"                        \
    "v_cmp_ne_u32 vcc, %[t1], %[si]\n\t"                       \
    "s_and_saveexec_b64 " lanes ", vcc\n\t"                    \
    "s_cbranch_execz vrt_kept%=\n\t"                           \
    "buffer_load_dwordx4 v[48:51], %[t1], %[rsec], 0 idxen\n\t" \
    "v_mov_b32 %[si], %[t1]\n"                                 \
    "vrt_kept%=:\n\t"                                          \
    "s_mov_b64 exec, " lanes "\n\t"
// The record, then the brick's mask bit (v53's sign) and the sector-level cell mask.
#define VRT_STEP_SECTOR(lanes) VRT_STEP_RECORD(lanes)          \
    "v_lshrrev_b32 %[t2], 1, %[g2]\n\t"                        \
    "v_lshrrev_b32 %[t0], 3, %[g0]\n\t"                        \
    "v_lshlrev_b32 %[t1], 1, %[g1]\n\t"                        \
    "v_bitop3_b32 %[t0], 12, %[t2], %[t0] bitop3:0xca\n\t"     \
    "v_bitop3_b32 %[t1], 48, %[t1], %[t0] bitop3:0x35\n\t"     \
    "v_bitop3_b32 %[t0], 16, %[g1], %[t0] bitop3:0xca\n\t"     \
    "v_and_b32 %[t0], 26, %[t0]\n\t"                           \
    "s_waitcnt vmcnt(0)\n\t"                                   \
    "v_lshlrev_b64 v[52:53], %[t1], v[48:49]\n\t"              \
    "v_cmp_gt_i32 vcc, 0, v53\n\t"                             \
    "v_lshrrev_b32 %[t0], %[t0], v51\n\t"                      \
    "v_bitop3_b32 %[cm], %[t0], 24, 7 bitop3:0xea\n\t"
// Lanes vcc are in an allocated brick or outside the world (the border's base slot is negative).
// The first look their 4x4x4 cell's mask up (v[52:53]; slot: their brick's slot + 1); t1 and t2
// are the voxel's shifts.  t2 is g2 >> 1 before.
#define VRT_STEP_CELL_LOAD                                     \
    "s_mov_b64 exec, vcc\n\t"                                  \
    "v_cmp_gt_i32 vcc, 0, v50\n\t"                             \
    "s_mov_b64 %[stop], vcc\n\t"                               \
    "s_andn2_b64 exec, exec, vcc\n\t"                          \
    "s_cbranch_execz vrt_stop%=\n\t"                           \
    "v_bcnt_u32_b32 %[slot], v52, 0\n\t"                       \
    "v_bcnt_u32_b32 %[slot], v53, %[slot]\n\t"                 \
    "v_and_b32 %[t1], 4, %[g1]\n\t"                            \
    "v_add_u32 %[slot], v50, %[slot]\n\t"                      \
    "v_bfe_u32 %[t0], %[g0], 2, 1\n\t"                         \
    "v_and_or_b32 %[t1], %[t2], 2, %[t1]\n\t"                  \
    "v_lshl_or_b32 %[t0], %[slot], 3, %[t0]\n\t"               \
    "v_or_b32 %[t0], %[t0], %[t1]\n\t"                         \
    "buffer_load_dwordx2 v[52:53], %[t0], %[rocc], 0 idxen\n\t" \
    "v_lshlrev_b32 %[t2], 2, %[g2]\n\t"                        \
    "v_lshlrev_b32 %[t1], 4, %[g1]\n\t"                        \
    "v_bitop3_b32 %[t2], 12, %[t2], %[g0] bitop3:0xca\n\t"     \
    "v_bitop3_b32 %[t1], 48, %[t1], %[t2] bitop3:0x35\n\t"     \
    "v_bitop3_b32 %[t2], %[t1], 42, %[t1] bitop3:0x0c\n\t"
// Then they stop at a solid voxel.
#define VRT_STEP_CELL VRT_STEP_CELL_LOAD                       \
    "s_waitcnt vmcnt(0)\n\t"                                   \
    "v_lshlrev_b64 v[54:55], %[t1], v[52:53]\n\t"              \
    "v_or_b32 %[t0], v52, v53\n\t"                             \
    "v_cmp_gt_i32 vcc, 0, v55\n\t"                             \
    "v_lshrrev_b64 v[54:55], %[t2], v[52:53]\n\t"              \
    "s_or_b64 %[stop], %[stop], vcc\n\t"                       \
    "v_and_b32 %[t1], 0x330033, v54\n\t"
// t0: the cell's mask, ored; t1: its 2x2x2 group's.  Cell mask 3 when the first is 0, 1 when the
// second is.  The lanes that stop note the step and leave exec.
#define VRT_STEP_STOP                                          \
    "v_sub_u32 %[t0], 1, %[t0] clamp\n\t"                      \
    "v_sub_u32 %[t1], 1, %[t1] clamp\n\t"                      \
    "v_lshl_or_b32 %[cm], %[t0], 1, %[t1]\n"                   \
    "vrt_stop%=:\n\t"                                          \
    "s_mov_b64 exec, %[stop]\n\t"                              \
    "v_mov_b32 %[iters], %[it]\n\t"                            \
    "s_andn2_b64 exec, %[alive], %[stop]\n\t"                  \
    "s_cbranch_execnz vrt_advance%=\n"
#define VRT_STEP_BRICK VRT_STEP_CELL "v_add_u32 %[desc], 1, %[desc]\n\t" VRT_STEP_STOP

// Operands of both loops (positions c, side distances s, directions d, 1 / d i, tStart ts, origin o,
// corner masks m, bias b, per axis).
#define VRT_STEP_OUT(C, S, G)                                                                                   \
    [c0] "+&v"(C[0]), [c1] "+&v"(C[1]), [c2] "+&v"(C[2]), [s0] "+&v"(S[0]), [s1] "+&v"(S[1]), [s2] "+&v"(S[2]), \
        [g0] "+&v"(G[0]), [g1] "+&v"(G[1]), [g2] "+&v"(G[2]), [iters] "+&v"(iters), [si] "+&v"(si),             \
        [slot] "+&v"(slot1), [it] "+&s"(it), [cm] "=&v"(cm), [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2),    \
        [base] "=&v"(base), [save] "=&s"(save), [alive] "=&s"(alive), [stop] "=&s"(stop)
#define VRT_STEP_IN(O, D, I, T, M, B, cap)                                                                      \
    [o0] "v"(O[0]), [o1] "v"(O[1]), [o2] "v"(O[2]), [d0] "v"(D[0]), [d1] "v"(D[1]), [d2] "v"(D[2]),             \
        [i0] "v"(I[0]), [i1] "v"(I[1]), [i2] "v"(I[2]), [ts0] "v"(T[0]), [ts1] "v"(T[1]), [ts2] "v"(T[2]),      \
        [m0] "v"(M[0]), [m1] "v"(M[1]), [m2] "v"(M[2]), [b0] "v"(B[0]), [b1] "v"(B[1]), [b2] "v"(B[2]),         \
        [max] "s"(cap), [sz] "s"(w.step_z), [sy] "s"(w.step_y), [sk] "v"(step_bias(w)), [rsec] "s"(rsec), [rocc] "s"(rocc)
#define VRT_STEP_CLOBBERS "v48", "v49", "v50", "v51", "v52", "v53", "v54", "v55", "vcc", "scc"

// The fast loop, for quick or guarded rays.
// GROUPS: a group word first says whether the sector is empty.  It spares a step in an empty
// sector the record (the word serves up to four sectors of a ray), for a second load that waits on
// the first in the others.
template <bool GROUPS>
__device__ __forceinline__ bool ray_trace_fast(const WorldView& w, RayState& r, uint32_t max_iters, int32_t v[3],
                                               uint32_t& slot, uint32_t first) {
    float bias[3];
#pragma unroll
    for (int a = 0; a < 3; a++) bias[a] = 8388608.0f + (float)(r.W[a] + kStepPad);
    uint32_t g[3];
    biased_floor(r.cur, bias, g);
    if (first == 0) {
        // a ray that starts outside the world misses at once; every other stays within the border
        uint32_t u[3];
#pragma unroll
        for (int a = 0; a < 3; a++) u[a] = g[a] - (0x4B000000u + (uint32_t)kStepPad);
        if (!((u[0] | u[2]) < w.size_xz && u[1] < w.size_y)) return false;
    }
    const i32x4 rsec = buffer_rsrc(w.steps, 16, w.step_n);
    // slot + 1 is what a step computes: the base is one slot (8 masks) early
    const i32x4 rocc = buffer_rsrc(w.occ - 8, 8, w.occ_n + 8u);
    uint32_t iters = max_iters, si = ~0u, slot1 = 0, base, it = first;
    uint32_t cm, t0, t1, t2;
    uint64_t save, alive, stop;
    if constexpr (GROUPS) {
        const i32x4 rgrp = buffer_rsrc(w.sgroups, 8, w.group_n);
        uint32_t gi = ~0u;
        uint64_t lanes;
        asm volatile("s_mov_b64 %[save], exec\n\t"
                     "s_branch vrt_look%=\n\t.p2align 6\n"
                     "vrt_back%=:\n\t"
                     "s_mov_b64 exec, %[alive]\n"
                     "vrt_advance%=:\n\t" VRT_STEP_ADVANCE("%[t0]", VRT_STEP_BIAS)
                     VRT_STEP_FLOOR "vrt_look%=:\n\t" VRT_STEP_GROUP VRT_STEP_SECTOR("%[lanes]")
                     "s_cbranch_vccz vrt_back%=\n\t" VRT_STEP_BRICK
                     "vrt_done%=:\n\t"
                     "s_mov_b64 exec, %[save]\n\t"
                     "v_mov_b32 %[base], v50"
                     : VRT_STEP_OUT(r.cur, r.side, g), [desc] "+&v"(r.descents), [gi] "+&v"(gi), [lanes] "=&s"(lanes)
                     : VRT_STEP_IN(r.o, r.d, r.inv, r.ts, r.dm, bias, max_iters), [gz] "s"(w.group_z), [gy] "s"(w.group_y), [rgrp] "s"(rgrp)
                     : VRT_STEP_CLOBBERS, "v56", "v57");
    } else {
        asm volatile("s_mov_b64 %[save], exec\n\t"
                     "s_branch vrt_look%=\n\t.p2align 6\n"
                     "vrt_advance%=:\n\t" VRT_STEP_ADVANCE("%[t0]", VRT_STEP_BIAS)
                     VRT_STEP_FLOOR "vrt_look%=:\n\t" VRT_STEP_SECTOR("%[alive]")
                     "s_cbranch_vccz vrt_advance%=\n\t" VRT_STEP_BRICK
                     "vrt_done%=:\n\t"
                     "s_mov_b64 exec, %[save]\n\t"
                     "v_mov_b32 %[base], v50"
                     : VRT_STEP_OUT(r.cur, r.side, g), [desc] "+&v"(r.descents)
                     : VRT_STEP_IN(r.o, r.d, r.inv, r.ts, r.dm, bias, max_iters)
                     : VRT_STEP_CLOBBERS);
    }
    const bool hit = iters < max_iters && (int32_t)base >= 0;
    v[0] = (int32_t)(g[0] & 0x7FFFFFu) - kStepPad;
    v[1] = (int32_t)(g[1] & 0x7FFFFFu) - kStepPad;
    v[2] = (int32_t)(g[2] & 0x7FFFFFu) - kStepPad;
    slot = slot1 - 1u;
    r.iters = iters + (hit ? 1u : 0u);
    return hit;
}

// RayCast's loop (CpuRenderer.cpp:185-202), a step at a time: until a hit, a miss or max_iters
// steps; true on a hit, with v the hit voxel and slot its brick slot.
// first: the steps the ray has already made (r.iters), for a ray resumed from a
// saved position and side distances; the loop then makes at most max_iters - first.
template <bool EXACT>
__device__ __forceinline__ bool ray_trace_steps(const WorldView& w, RayState& r, uint32_t max_iters, int32_t v[3],
                                                uint32_t& slot, uint32_t first) {
    bool hit = false;
    for (uint32_t it = first; it < max_iters; it++)
        if (!ray_advance<EXACT>(w, r, v, hit, &slot)) break;
    return hit;
}

// The cast of a wave's rays (set up by ray_setup): the fast loop when it is exact for all of them.
// One direction in 10^4 or so has a component too small for it, so a launch of some hundred waves has one
// that steps, and ends with it: tame rays take the shorter form, and ray_is_quick goes as far as the
// border allows.  50 k rays without order in the 2048^3 spheres: 82 us with the exact form and a
// quarter of that bound, 80 with the tame one, 74.6 with both.
template <bool GROUPS = false>
__device__ __forceinline__ bool ray_trace_wave(const WorldView& w, RayState& r, uint32_t max_iters, int32_t v[3],
                                               uint32_t& slot, uint32_t first = 0) {
    const bool near = origin_is_guarded(r.W) && masks_in_reach(w);  // uniform
    if (!(near && __all(ray_is_quick(r.o, r.d, r.inv)))) {
        ray_exact_inverse(r);
        const bool tame = __all(ray_is_tame(r));
        if (!(near && tame && __all(ray_is_guarded(w, r))))
            return tame ? ray_trace_steps<false>(w, r, max_iters, v, slot, first)
                        : ray_trace_steps<true>(w, r, max_iters, v, slot, first);
    }
    return ray_trace_fast<GROUPS>(w, r, max_iters, v, slot, first);
}

// Hit record fields (vrt_hit in vrt.h) of a finished ray.
__device__ __forceinline__ void ray_hit_record(const WorldView& w, const RayState& r, const int32_t v[3],
                                               uint32_t slot, float& t, int4& rec) {
    float tt = min_x86(min_x86(r.side[0], r.side[1]), r.side[2]);
    bool X = r.side[0] == tt, Y = r.side[1] == tt, Z = !X && !Y;
    uint32_t code = (X ? (signbit(r.d[0]) ? 1u : 3u) : 0u) | (Y ? (signbit(r.d[1]) ? 1u : 3u) : 0u) << 2 |
                    (Z ? (signbit(r.d[2]) ? 1u : 3u) : 0u) << 4;
    uint32_t ux = (uint32_t)v[0], uy = (uint32_t)v[1], uz = (uint32_t)v[2];
    uint32_t mat = w.vox[(size_t)slot * 512 + ((ux & 7u) | (uz & 7u) << 3 | (uy & 7u) << 6)];
    t = tt;
    rec = make_int4(v[0], v[1], v[2], (int)(mat | code << 8 | (r.iters & 0xFFFFu) << 16));
}

__device__ __forceinline__ void ray_miss_record(const RayState& r, float& t, int4& rec) {
    t = -1.0f;
    rec = make_int4(0, 0, 0, (int)((r.iters & 0xFFFFu) << 16));
}

}  // namespace vrt
