// launch_uneven.hpp -- host-side interface of the persistent uneven-batch
// kernel (uneven.hip) and its plan (capi.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace tprh {

// Slice shapes the persistent kernel carries a code path for: (id, E, L).
// Its 1024-lane workgroups leave 128 VGPRs per lane, so the menu stops at
// the shapes whose fast path fits (E = 16 with L > 16 and E = 32 need more);
// every size class up to n = 16384 has a shape here (s = 256, E = L = 16).
#define TPRH_UNEVEN_SHAPES(X) \
    X(0, 1, 16)               \
    X(1, 2, 16)               \
    X(2, 4, 16)               \
    X(3, 8, 16)               \
    X(4, 16, 16)              \
    X(5, 8, 32)               \
    X(6, 4, 64)               \
    X(7, 8, 64)

inline int uneven_shape_id(int E, int L) {
#define TPRH_UNEVEN_ID(ID, EE, LL) \
    if (E == EE && L == LL) return ID;
    TPRH_UNEVEN_SHAPES(TPRH_UNEVEN_ID)
#undef TPRH_UNEVEN_ID
    return -1;
}

// Lanes of a workgroup, and so of an item.  Where every system of a plan (or
// serving batch) fits 256 lanes (n = 4096 at 16 equations per lane), 256, one
// item per workgroup: four workgroups to a CU load, solve and store in turn,
// and a small plan covers four times the CUs; no counter, no launch to clear
// it.  Else 1024 for all, in a persistent kernel.  Measured, fast PTPR, all in
// 1024 -> in 256: 150 systems of 512 .. 2048 15.7 -> 6.4 us, 10000 of 128 ..
// 1024 32.0 -> 17.5.  The larger systems in 1024 and the others in a second
// launch of 256 is slower: 1249 of 512 .. 16384 50 us against 42.5, 20000 of
// 256 .. 16384 396 against 388.
constexpr int kSlotTile = 256;
constexpr int kSlotBig = 1024;
constexpr int slot_block(int most) { return most <= kSlotTile ? kSlotTile : kSlotBig; }

// LDS of a workgroup: an item holds block / (m L) systems of 13 m floats
// each, at most 13 * block / 16 floats for any shape of the menu, and behind
// them, where loads, stores or equations are turned through LDS
// (solve_slot.hpp), 17 floats per lane.
constexpr int slot_row_words(int block) { return 13 * block / 16; }
constexpr size_t slot_lds_bytes(int block, bool turned) {
    return sizeof(float) * ((size_t)slot_row_words(block) + (turned ? (size_t)block * 17 : 0));
}
// The 1024-lane kernels turn in exact PTPR only.
constexpr size_t slot_big_lds(int method, int mode) { return slot_lds_bytes(kSlotBig, method == 0 && mode == 1); }

// One work item: `count` systems of one size class, as many as one workgroup
// holds (block / (m * L)).
struct UnevenTask {
    int shape;     // TPRH_UNEVEN_SHAPES id
    int m;         // slices per system
    int lg_lanes;  // log2(m * L): lanes per system
    int first;     // first entry of the plan's system list
    int count;     // systems in the item
};

struct UnevenLaunch {
    const UnevenTask* tasks;
    int ntasks;
    int block;     // lanes of a workgroup
    int* counter;  // of the persistent kernel
    const int* sys_list;
    const long long* offsets;
    const float *a, *b, *c, *d;
    float* x;
    int grid;  // workgroups of the persistent kernel
};

hipError_t launch_uneven(int method, int mode, const UnevenLaunch& p, hipStream_t stream);
// Workgroups of 1024 lanes per CU.
hipError_t uneven_occupancy(int method, int mode, int* blocks_per_cu);

}  // namespace tprh
