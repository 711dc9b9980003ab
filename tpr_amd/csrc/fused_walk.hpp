// fused_walk.hpp -- what a workgroup of the one-pass form (split_fused.hpp)
// does next: its own tiles first, then those it had to put aside, and in
// between the tiles that others have not published.  Host and device code
// alike, so that a CPU test can run the same decisions for many sets of
// workgroups of which only some are there.
#pragma once
#include <hip/hip_runtime.h>

namespace tprh {

constexpr int kFusedGroup = 16;  // tiles per group (one DPP row)

// A workgroup's next task: a tile of its own, one of its own taken up again,
// or one of another workgroup published on its behalf.
enum FusedKind { kFusedOwn = 0, kFusedAgain = 1, kFusedHelp = 2 };

// One of the set bits of `missing`: the first from bit `from` on, or else the
// first of all, so that workgroups which wait for the same blocks start on
// different ones.
__host__ __device__ inline int fused_pick(unsigned long long missing, int from) {
    const unsigned long long above = missing >> from << from;
    return __builtin_ctzll(above ? above : missing);
}

// Systems of more than 16 tiles, for a workgroup that has waited for tile ti
// in vain: -1 once every tile and every group is published, else a tile (in
// the system) that was missing when it was looked at.  x.tiles(g, limit) and
// x.groups(limit) poll up to `limit` more times for the 16 tiles of group g
// and for the groups, and return which are missing; x.publish(g) publishes
// group g from the tiles just read: a group whose tiles are all there, but
// whose first tile's workgroup is not, is published here.
template <typename X>
__host__ __device__ __forceinline__ int fused_look(X& x, int ti, int limit) {
    const int own = ti / kFusedGroup;
    for (int g = own;;) {  // ends: each turn publishes a missing group
        unsigned long long m = x.tiles(g, limit);
        if (m != 0) return g * kFusedGroup + fused_pick(m, ti % kFusedGroup);
        x.publish(g);
        m = x.groups(limit);
        if (m == 0) return -1;
        g = fused_pick(m, own);
        limit = 0;
    }
}

// Whether a workgroup publishes the tile it has loaded.  seen: the tile was
// published already when its loads were complete (asked for on behalf of
// another workgroup only).  The answers of a system are stored once all its
// tiles are published, so what was loaded before that are its inputs, even
// where x is stored over d; after it, they may not be, and the words are there.
__host__ __device__ inline bool fused_publishes(int kind, bool seen) {
    return kind == kFusedOwn || (kind == kFusedHelp && !seen);
}

// Tasks that a workgroup can need beyond its own tiles, of which it has at
// most total / stride, rounded up: each is taken up again, all other tiles of
// its system are published, it is taken up once more; at the end there is no
// tile left.  Only words or lists that something else changes (two
// overlapping solves in one workspace) can make it need more.
__host__ __device__ inline int fused_task_limit(int total, int stride, int bps) {
    return ((total + stride - 1) / stride) * (bps + 2) + 1;
}

struct FusedTask {
    int tile;  // -1: the workgroup is done
    int kind;
};

// The lists of one workgroup, kept by its thread 0: tiles of its own whose
// system was not all there in time (linked through the workspace), and those
// taken up again in vain.
struct FusedWalk {
    int head = -1, again = -1;
    int tries = 0;  // tasks beyond its own tiles

    // Past `limit` tasks (fused_task_limit) no tile is waited for or helped
    // with any more: the caller answers one taken up again in vain with NaN,
    // as if all were there.  limit: no less than the workgroup's own tiles.
    __host__ __device__ __forceinline__ bool lost(int limit) const { return tries > limit; }

    // After task (tile, kind): ok, the system was all there (and an own
    // tile's x is stored); missing, a tile of it that was not.  own: the
    // workgroup's next own tile, -1 when it has none left.  A tile taken up
    // again in vain is followed by help with one missing tile after the
    // other until its system is all there.
    template <typename Link>
    __host__ __device__ __forceinline__ FusedTask next(int tile, int kind, bool ok, int missing, int own, int limit,
                                                       Link&& link) {
        if (!ok && kind != kFusedHelp) {
            int& to = kind == kFusedOwn ? head : again;
            link(tile) = to;
            to = tile;
        }
        if (own >= 0) return {own, kFusedOwn};
        if (tries > 2 * limit + 2) return {-1, kFusedAgain};  // a list without an end
        tries++;
        if (!ok && kind != kFusedOwn && tries <= limit) return {missing, kFusedHelp};
        if (head < 0) {
            head = again;
            again = -1;
        }
        const int t = head;
        if (t >= 0) head = link(t);
        return {t, kFusedAgain};
    }
};

}  // namespace tprh
