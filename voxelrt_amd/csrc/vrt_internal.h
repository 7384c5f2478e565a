// vrt_internal.h - shared internals of libvoxelrt_hip.so (not part of the ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "vrt.h"

namespace vrt {

// ---------------------------------------------------------------- errors

void set_error(const std::string& msg);
void clear_error();

// Returns a vrt_status after recording the message.
int fail(int status, const std::string& msg);
int hip_fail(hipError_t e, const char* what);

#define VRT_HIP(call)                                     \
    do {                                                  \
        hipError_t e_ = (call);                           \
        if (e_ != hipSuccess) return ::vrt::hip_fail(e_, #call); \
    } while (0)

// Wraps a body so that no C++ exception crosses the ABI.
template <typename F>
int guarded(F&& f) {
    try {
        clear_error();
        return f();
    } catch (const std::bad_alloc&) {
        return fail(VRT_ERR_CAPACITY, "host allocation failed");
    } catch (const std::exception& ex) {
        return fail(VRT_ERR_STATE, ex.what());
    } catch (...) {
        return fail(VRT_ERR_STATE, "unknown exception");
    }
}

// Test hook: VRT_FAULT_INJECT=<entry name> makes that entry report a HIP error.
bool fault_injected(const char* entry);

// ---------------------------------------------------------------- slot arena

// Largest slot arena of a world.
constexpr uint64_t kMaxSlots = 1ull << 28;


// Free-list arena of brick slots.  Each sector owns one contiguous run of
// popcount(mask) slots.  Slot 0 is valid (no sentinel).  Best-fit allocation,
// growth in place when the following range is free, coalescing on free.
class SlotArena {
public:
    explicit SlotArena(uint32_t capacity = 0) : capacity_(capacity) {
        if (capacity) free_[0] = capacity;
    }
    // Moves/grows a run from (base, cur) to a run of `want` slots. Returns false when full.
    bool realloc(uint32_t& base, uint32_t cur, uint32_t want);
    void release(uint32_t base, uint32_t size);
    uint32_t allocated() const { return allocated_; }
    uint32_t capacity() const { return capacity_; }
    size_t free_ranges() const { return free_.size(); }
    // One past the highest allocated slot.
    uint32_t high_water() const;

private:
    std::map<uint32_t, uint32_t> free_;  // start -> length
    uint32_t capacity_ = 0;
    uint32_t allocated_ = 0;
};

// ---------------------------------------------------------------- device world view

// Sector record in HBM (vrt_sector_record in vrt.h): allocation mask (lo, hi), base
// slot, and the cell mask of a step at the sector level whose 2x2x2 group of bricks
// is empty: 15 (a 16-voxel cell), or 31 (the whole sector) when the mask is 0, the
// reference's +2 LOD of an empty mask; a step whose group holds a brick uses half.
__host__ __device__ inline uint4 sector_record(uint64_t mask, uint32_t base) {
    return make_uint4((uint32_t)mask, (uint32_t)(mask >> 32), base, mask ? 15u : 31u);
}

// What the fast step reads (ray_trace_fast): two tables over the world and a border around it, so a
// step that leaves the world lands in the border and needs no bounds test.  Their indices come
// from padded coordinates, the voxel's plus kStepPad (one group of 4x4x4 sectors) on each axis.
constexpr int32_t kStepPad = 128;
constexpr uint32_t kStepFirst = 3;
// The group table: per group of 4x4x4 sectors a u64, bit x | z << 2 | y << 4 set when that sector
// has a brick or lies outside the world.  Group (X, Y, Z) of the padded coordinates (>> 7) is word
// X + Z * group_z + Y * group_y.
// The step table: per sector a 16-byte record, and border records around them: one sector before the
// world, and after it up to one past the world's last sector or the group of 4, whichever is
// further (the shader method's cells are up to a group wide).
// Sector (X, Y, Z) of the padded coordinates (>> 5; the world's first is 4, the border's kStepFirst) is
// record X - kStepFirst + (Z - kStepFirst) * step_z + (Y - kStepFirst) * step_y.
//   x, y  allocation mask; all ones in the border (the step's brick test then succeeds)
//   z     base slot; all ones in the border (base slots are below 2^28)
//   w     per 2x2x2 group of bricks (gx, gz, gy = bit 4 of x, z, y) the cell mask of a step that
//         stays at the sector level: bits 3..4 of w >> (2 gx + 8 gz + 16 gy) are bits 3..4 of that
//         mask, whose bits 0..2 are always set: 7 when the group holds a brick, 15 when it is
//         empty, 31 when the sector is.  Bits 8..9 are the shader method's level above an empty
//         sector (group_lod), 0 otherwise
__host__ __device__ inline uint4 step_record(uint64_t mask, uint32_t base) {
    uint32_t codes = 0;
    for (uint32_t g = 0; g < 8; g++) {
        const uint32_t gx = g & 1u, gz = (g >> 1) & 1u, gy = g >> 2;
        const uint64_t group = (uint64_t)0x00330033u << (2 * gx + 8 * gz + 32 * gy);
        const uint32_t code = mask == 0 ? 3u : ((mask & group) == 0 ? 1u : 0u);
        codes |= code << (3 + 2 * gx + 8 * gz + 16 * gy);
    }
    return make_uint4((uint32_t)mask, (uint32_t)(mask >> 32), base, codes);
}
// The shader method steps 32, 64 or 128 voxels over an empty sector: 128 when the mask of its 4x4x4
// sectors is 0, 64 when its 2x2x2 group of them is.  Code 0, 1 or 3 for sector x | z << 2 | y << 4:
// bits 5..6 of the cell mask.
__host__ __device__ inline uint32_t group_lod(uint64_t group, uint32_t sector) {
    const uint32_t half = sector < 32 ? (uint32_t)group : (uint32_t)(group >> 32);
    return group == 0 ? 3u : (((half >> (sector & 0xAu)) & 0x00330033u) == 0 ? 1u : 0u);
}
// The mask table: the step table's records by index, as the ray-cell table (ShaderView) needs them.
//   x, y  allocation mask; of an empty sector its group's mask, in which its own bit is 0, so
//         the step's brick test fails there too; all ones in the border
//   z     base slot; all ones in the border
//   w     log2 of the voxels per bit of that mask: 3, or 5 for an empty sector
__host__ __device__ inline uint4 mask_record(uint64_t mask, uint32_t base, uint64_t group) {
    const uint64_t m = mask ? mask : group;
    return make_uint4((uint32_t)m, (uint32_t)(m >> 32), base, mask ? 3u : 5u);
}
inline __host__ __device__ uint4 step_border_record() { return make_uint4(~0u, ~0u, ~0u, 0u); }

struct WorldView {
    const uint4* __restrict__ sec;       // [nsec]
    const uint4* __restrict__ steps;     // [step_n] the step table
    const uint64_t* __restrict__ sgroups;  // [group_n] the group table
    uint32_t step_z, step_y, step_n;     // their strides and sizes in records
    uint32_t group_z, group_y, group_n;
    const uint64_t* __restrict__ occ;    // [occ_n], slots * 8
    uint32_t occ_n;
    const uint8_t* __restrict__ vox;     // [slots * 512]
    uint32_t size_xz, size_y;            // voxel extents
    uint32_t shift_xz, shift_y;          // log2 sector grid extents
};

// What the shader method reads beyond WorldView: the sector-of-sectors masks
// (one u64 per 4x4x4 group of sectors, bit = that sector has a brick; group grid
// of max(1, sectors / 4) per axis) and the ray-cell interaction table.
struct ShaderView {
    WorldView w;
    const uint64_t* __restrict__ groups;  // [1 << (2 * gshift_xz + gshift_y)]
    const uint4* __restrict__ masks;      // [w.step_n] the mask table
    const uint64_t* __restrict__ lut;     // [8 octants * 64 cells]
    uint32_t gshift_xz, gshift_y;
};

// Ray-cell interaction table: for direction octant oct (bit a set = positive
// along axis a) and cell c of a 4x4x4 mask, the cells c + j * dir (j >= 0 per
// axis) inside the mask, i.e. the cells a ray in that octant can reach from c.
void ray_cell_lut(uint64_t table[512]);

}  // namespace vrt

struct vrt_world {
    int device = 0;
    uint32_t log2_xz = 0, log2_y = 0;
    uint32_t shift_xz = 0, shift_y = 0;
    uint32_t nsec = 0;
    uint8_t* d_tables = nullptr;      // one allocation for every table but d_occ and d_vox
    uint4* d_sec = nullptr;           // packed sector records (mask, base slot)
    uint4* d_steps = nullptr;         // the step table
    uint4* d_masks = nullptr;         // the mask table
    uint64_t* d_sgroups = nullptr;    // the group table
    uint64_t* d_occ = nullptr;
    uint8_t* d_vox = nullptr;
    uint64_t* d_palette = nullptr;
    uint32_t slot_cap = 0;            // device slots backed by memory
    std::vector<uint64_t> h_mask;     // host mirror of the sector headers
    std::vector<uint32_t> h_base;
    vrt::SlotArena arena;
    uint32_t num_bricks = 0;
    uint32_t full_sectors = 0;        // sectors that hold a brick
    // shader method: sector-of-sectors masks and the ray-cell table
    uint32_t gshift_xz = 0, gshift_y = 0;
    std::vector<uint64_t> h_groups;
    uint64_t* d_groups = nullptr;
    uint64_t* d_lut = nullptr;
    // bumped whenever d_occ / d_vox move (slot growth): device pointers taken earlier, e.g. in a
    // captured graph, are stale once it changes
    uint32_t generation = 0;
    // set when a sync fails after its device work began: the device tables may then disagree
    // with the host mirror, and every later call on the world returns VRT_ERR_STATE
    bool failed = false;
    // sync staging, owned by the world and reused by every sync: two pinned host halves and two
    // device halves of kSyncHalf bytes (a chunk is packed into one half while the other's copy
    // and apply kernel run); stage_ev[h] is recorded after the last kernel that reads half h
    uint8_t* h_stage = nullptr;
    uint8_t* d_stage = nullptr;
    hipEvent_t stage_ev[2] = {nullptr, nullptr};
    bool stage_pending[2] = {false, false};
    uint32_t stage_next = 0;
    // bricks whose slot changes while their contents stay: gathered here, then written back
    uint8_t* d_moves = nullptr;
    size_t moves_cap = 0;
    hipEvent_t moves_ev = nullptr;
    bool moves_pending = false;
    // picking: the host memory its kernel writes its result to, and the last pick's number
    void* h_pick = nullptr;
    mutable std::mutex pick_mu;
    mutable uint32_t pick_seq = 0;
    // totals since creation
    uint64_t upload_bytes = 0, upload_brick_bytes = 0, moved_bricks = 0;

    // at least 4 sectors a side and the border
    uint32_t step_z() const { return std::max(4u, 1u << shift_xz) + 2u; }
    uint32_t step_y() const { return step_z() * step_z(); }
    uint32_t step_n() const { return step_y() * (std::max(4u, 1u << shift_y) + 2u); }
    uint32_t group_z() const { return (1u << gshift_xz) + 2u; }
    uint32_t group_y() const { return group_z() * group_z(); }
    uint32_t group_n() const { return group_y() * ((1u << gshift_y) + 2u); }
    // the bits of a group word past the end of a world of fewer than 4 sectors on an axis
    uint64_t group_outside() const {
        uint64_t m = 0;
        for (uint32_t b = 0; b < 64; b++)
            if ((b & 3u) >> shift_xz || ((b >> 2) & 3u) >> shift_xz || (b >> 4) >> shift_y) m |= 1ull << b;
        return m;
    }

    vrt::WorldView view() const {
        vrt::WorldView v;
        v.sec = d_sec;
        v.steps = d_steps;
        v.step_z = step_z();
        v.step_y = step_y();
        v.step_n = step_n();
        v.sgroups = d_sgroups;
        v.group_z = group_z();
        v.group_y = group_y();
        v.group_n = group_n();
        v.occ = d_occ;
        v.occ_n = slot_cap * 8u;
        v.vox = d_vox;
        v.size_xz = 1u << log2_xz;
        v.size_y = 1u << log2_y;
        v.shift_xz = shift_xz;
        v.shift_y = shift_y;
        return v;
    }
    vrt::ShaderView shader_view() const {
        vrt::ShaderView v;
        v.w = view();
        v.groups = d_groups;
        v.masks = d_masks;
        v.lut = d_lut;
        v.gshift_xz = gshift_xz;
        v.gshift_y = gshift_y;
        return v;
    }
};

namespace vrt {
// Bytes of a world's picking result.
constexpr size_t kPickBytes = 64;
// Bytes of one sync staging half (host pinned and device).
constexpr size_t kSyncHalf = (size_t)8 << 20;

// Blocks of the next launch of a kernel that needs `left` more: a launch has fewer than 2^32 lanes.
inline uint32_t launch_blocks(uint64_t left, uint32_t threads) {
    return (uint32_t)std::min<uint64_t>(left, 0xFFFFFFFFu / threads);
}

// VRT_OK, or VRT_ERR_STATE (with the message) when a failed sync left the world unusable.
int check_world(const vrt_world* w, const char* entry);
}  // namespace vrt
