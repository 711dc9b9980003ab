// split_fused.hpp -- fast PTPR on systems larger than one workgroup in one
// pass: every equation is read once and x written once (20 B/eq), against 36
// B/eq for the two passes of split_kernels.hpp.
//
// What bounds it: HBM.  The two passes move 604 MB for 256 x N=65536 at the
// rate such bytes can be moved (K1 46, K2 6, K3 47 us); reading the inputs
// once leaves 336 MB.  A whole solve of that batch: 101 us two passes, 65 us
// this way (5.1 TB/s; a device copy of that size reaches 4.8-5.4); with an
// fp16-stored solve and a refinement step 203 -> 134 us; one system of 1 Mi
// equations 29 -> 21 us.
//
// A tile is 4096 consecutive equations of one system: 256 lanes x 16, sixteen
// rows of 16 lanes (one DPP row, 256 equations).  A workgroup
//   1. loads its tile and runs the two-level stage 1 on every row
//      (fast16_stage1), which leaves each row's first and last unknown in
//      terms of the unknowns just outside the row;
//   2. reduces its sixteen rows to two equations, of the tile's first and
//      last unknown, in terms of the unknowns just outside the tile: the E_st
//      update and the reduced rows of src/ptpr.cpp:193-241, then four DPP
//      levels of PCR, in every DPP row redundantly so that no wavefront waits
//      for another;
//   3. publishes those six numbers, and waits for the other tiles' of its
//      system with its equations' state still in registers;
//   4. solves the system of the tiles' last unknowns by the same steps (one
//      tile per lane) and finishes its rows from the unknowns on either side
//      of the tile (src/ptpr.cpp:263-287, x[ed+1] from the next row's first
//      equation instead of a division by c_ed).
// So one exchange of 24 bytes per 4096 equations crosses the chip, and the
// only wait is for the slowest tile of the system.  It needs no fence and no
// counter: the words are device-coherent, set to a NaN pattern that is never
// published before the launch (clear_fused_kernel), and a reader polls until
// no word of that pattern is left.  Four workgroups live on a CU at once, so
// that one's wait (4.3 us of a tile's 12 at the median) is covered by others'
// loads.
//
// Slices: s = 256 (one row), 512, 1024 or 2048 (several rows) -- in fast
// arithmetic a slice's interior, and the rows of a tile, may be eliminated in
// any order.
//
// The solve ends whichever workgroups are resident.  Workgroup k of a grid of
// G takes tiles k, k + G, ...; it publishes a tile before it waits, and waits
// only `spin` polls: then it puts the tile on a list (linked through the
// workspace) and goes on with its next one.  Its own tiles done, it takes the
// listed ones up again (loading them again); where one still misses a tile,
// that tile's workgroup may not have started, and it computes and publishes
// the missing tile on that workgroup's behalf (the same words), so each
// workgroup can finish with no other's help.  With a grid that the device
// holds at once, as launched here, on an otherwise idle device, no tile is
// ever listed.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

#include "split_kernels.hpp"

namespace tprh {

constexpr int kFusedTile = 4096;               // equations per workgroup
constexpr int kFusedThreads = 256;
constexpr int kFusedGroup = 16;                // tiles per group (one DPP row)
constexpr int kFusedWave = 64;                 // blocks of a chain that one wavefront solves
constexpr unsigned kFusedEmpty = 0xffffffffu;  // a word not yet published
constexpr int kFusedSpin = 64;                 // polls (about a microsecond each) before a tile is listed
constexpr int kFusedTries = 1 << 14;           // tasks of one workgroup beyond its own tiles, in all

// A workgroup's next task: a tile of its own, one of its own taken up again,
// or one of another workgroup published on its behalf.
enum FusedKind { kFusedOwn = 0, kFusedAgain = 1, kFusedHelp = 2 };

// A system's boundary buffer (Rows) of bps tiles holds: words 8 t .. 8 t + 7
// what tile t publishes, its equations [F.a, F.c, F.r, L.a, L.c, L.r] (F:
// first unknown, L: last) and, with refinement, the iterate's x at both; from
// 8 bps one word per tile, the list link; from 9 bps eight words per group of
// 16 tiles, its equations.  9.5 words per tile in all; the buffer has 8 per
// slice, two slices or more per tile.
__device__ __forceinline__ int* fused_link(float* rows, int bps, int t) {
    return reinterpret_cast<int*>(rows) + 8 * (size_t)bps + t;
}
__device__ __forceinline__ float* fused_groups(float* rows, int bps) { return rows + 9 * (size_t)bps; }

// Marks every published word empty: one thread per tile (a kernel, not a
// memset, so that a captured graph replays it).
template <typename Loc>
__global__ __launch_bounds__(256) void clear_fused_kernel(Loc loc, int nsys, int lg_bps) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nsys << lg_bps) return;
    const int bps = 1 << lg_bps;
    const int t = i & (bps - 1);
    float* rows = loc.Rows(i >> lg_bps);
    const uint4 e = make_uint4(kFusedEmpty, kFusedEmpty, kFusedEmpty, kFusedEmpty);
    uint4* w = reinterpret_cast<uint4*>(rows + 8 * (size_t)t);
    w[0] = e;
    w[1] = e;
    if (bps > kFusedWave && t % kFusedGroup == 0) {
        w = reinterpret_cast<uint4*>(fused_groups(rows, bps) + 8 * (t / kFusedGroup));
        w[0] = e;
        w[1] = e;
    }
}

// Equations of the first and last unknown of a block (a row, a tile, a group)
// in terms of the unknowns just outside it:
//   x_first + fa x_before + fc x_after = fr,  x_last + la x_before + lc x_after = lr.
struct BlockEnds {
    float fa, fc, fr, la, lc, lr;
};

// Two floats as published (a NaN of the empty pattern becomes another NaN),
// and back; missing: not published yet.
__device__ __forceinline__ void publish_pair(float* p, float x, float y) {
    unsigned a = __builtin_bit_cast(unsigned, x), b = __builtin_bit_cast(unsigned, y);
    a = a == kFusedEmpty ? 0x7fffffffu : a;
    b = b == kFusedEmpty ? 0x7fffffffu : b;
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), (unsigned long long)b << 32 | a, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long read_pair(const float* p) {
    return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool pair_missing(unsigned long long v) {
    return (unsigned)v == kFusedEmpty || (unsigned)(v >> 32) == kFusedEmpty;
}
__device__ __forceinline__ float pair_first(unsigned long long v) { return __builtin_bit_cast(float, (unsigned)v); }
__device__ __forceinline__ float pair_second(unsigned long long v) {
    return __builtin_bit_cast(float, (unsigned)(v >> 32));
}

__device__ __forceinline__ void publish_ends(float* p, const BlockEnds& e) {
    publish_pair(p, e.fa, e.fc);
    publish_pair(p + 2, e.fr, e.la);
    publish_pair(p + 4, e.lc, e.lr);
}
// False while a word is missing.
__device__ __forceinline__ bool read_ends(const float* p, BlockEnds& e) {
    const unsigned long long v0 = read_pair(p), v1 = read_pair(p + 2), v2 = read_pair(p + 4);
    e = BlockEnds{pair_first(v0), pair_second(v0), pair_first(v1), pair_second(v1), pair_first(v2), pair_second(v2)};
    return !pair_missing(v0) && !pair_missing(v1) && !pair_missing(v2);
}

// Polls until lanes with `need` have read their blocks' words at p into
// their e; after `limit` polls gives up.  Returns the lanes still missing
// theirs.  Every lane of the wavefront calls this.
__device__ __forceinline__ unsigned long long wait_ends(const float* p, bool need, int limit, BlockEnds& e) {
    for (int i = 0;; i++) {
        if (need) need = !read_ends(p, e);
        const unsigned long long missing = __ballot(need);
        if (missing == 0 || i >= limit) return missing;
        __builtin_amdgcn_s_sleep(1);
    }
}

// A chain of 16 blocks, one per lane of a DPP row, reduced to the unknowns
// outside the row (x before lane 0's block, x after lane 15's): the E_st
// update (src/ptpr.cpp:193-211), the reduced rows (:218-241) and PCR on them.
struct Chain16 {
    float ta, tr, s1;  // x_first + ta x_before + s1 x_last = tr
    float pA, pC, pR;  // x_last = pR - pA x_outer_before - pC x_outer_after

    __device__ __forceinline__ void reduce(const BlockEnds& e, int l) {
        s1 = (fabsf(e.lc) < FLT_EPSILON) ? -1.0f : -e.fc / e.lc;
        ta = __builtin_fmaf(s1, e.la, e.fa);
        tr = __builtin_fmaf(s1, e.lr, e.fr);
        // the next block's first equation (past the row: x_after itself)
        const float na = shift_down<16, 1>(ta, 0.0f, l);
        const float nc = shift_down<16, 1>(s1, -1.0f, l);
        const float nr = shift_down<16, 1>(tr, 0.0f, l);
        const float inv = recip_rn(__builtin_fmaf(-na, e.lc, 1.0f));
        float Ap[1] = {-(inv * e.la)};
        float Cp[1] = {(inv * e.lc) * nc};
        float Rr[1] = {inv * __builtin_fmaf(-e.lc, nr, e.lr)};
        ptpr_stage1_fast16<1, 1>(Ap, Cp, Rr);
        pA = -Ap[0];
        pC = -Cp[0];
        pR = Rr[0];
    }
    // The chain's own ends, in every lane of its row (the row's lanes
    // `first` and first + 15 of the wavefront).
    __device__ __forceinline__ BlockEnds ends(int first) const {
        BlockEnds e;
        e.fa = __shfl(__builtin_fmaf(-s1, pA, ta), first, 64);
        e.fc = __shfl(-(s1 * pC), first, 64);
        e.fr = __shfl(__builtin_fmaf(-s1, pR, tr), first, 64);
        e.la = __shfl(pA, first + 15, 64);
        e.lc = __shfl(pC, first + 15, 64);
        e.lr = __shfl(pR, first + 15, 64);
        return e;
    }
    // From the unknowns outside the row: x just before the lane's block, its
    // last x and x just after it.
    __device__ __forceinline__ void solve(float before, float after, int l, float& xb, float& xe, float& xa) const {
        xe = __builtin_fmaf(-pC, after, __builtin_fmaf(-pA, before, pR));
        xb = shift_up<16, 1>(xe, before, l);
        const float xf = __builtin_fmaf(-s1, xe, __builtin_fmaf(-ta, xb, tr));
        xa = shift_down<16, 1>(xf, after, l);
    }
};

// A whole system of up to 64 blocks, one per lane (lanes past the last one
// hold zero equations): x just before and just after block k (uniform).
__device__ __forceinline__ void solve_blocks(const BlockEnds& e, int count, int k, int lane, float& before,
                                             float& after) {
    const int l = lane & 15;
    Chain16 c;
    c.reduce(e, l);
    float ob = 0.0f, oa = 0.0f;  // x outside the lane's row
    if (count > 16) {
        // the (at most four) rows' ends, row r in lane r of every row
        BlockEnds u = c.ends(lane & 48);
        auto gather = [&](float v) {
            const float w = __shfl(v, (l & 3) << 4, 64);  // every lane takes part
            return l < 4 ? w : 0.0f;
        };
        u = BlockEnds{gather(u.fa), gather(u.fc), gather(u.fr), gather(u.la), gather(u.lc), gather(u.lr)};
        Chain16 t;
        t.reduce(u, l);
        float xb, xe, xa;
        t.solve(0.0f, 0.0f, l, xb, xe, xa);
        const int src = (lane & 48) + (lane >> 4);
        ob = __shfl(xb, src, 64);
        oa = __shfl(xa, src, 64);
    }
    float xb, xe, xa;
    c.solve(ob, oa, l, xb, xe, xa);
    before = __shfl(xb, k, 64);
    after = k + 1 < count ? __shfl(xa, k, 64) : 0.0f;
}

// WIDE: more than kFusedWave tiles per system (up to 1024): the exchange is
// in two steps, the tiles of a group of 16 first, the groups then, so that a
// tile reads 16 + bps / 16 blocks' words instead of bps.
template <bool HAS_B, typename CT, bool REFINE, bool WIDE, typename Loc>
__global__ __launch_bounds__(kFusedThreads, REFINE ? 3 : 4) void fused_split_kernel(Loc loc, int nsys, int lg_bps, int first,
                                                                                    int stride, int spin) {
    constexpr int E = 16;
    __shared__ __align__(16) float stage_lds[stage_words<E>(kFusedThreads)];
    __shared__ float s_ends[6][16];  // E_st and E_ed of the tile's rows
    __shared__ float s_side[2];      // x just before and just after the tile
    __shared__ int s_seen[4];        // per wavefront: the tile was published before it was loaded
    __shared__ float s_xlast;        // the iterate's last x of the tile
    __shared__ int s_ok, s_tile, s_kind;
    const int bps = 1 << lg_bps;
    const int total = nsys << lg_bps;
    const int lane = threadIdx.x & 63;
    const int l = threadIdx.x & 15;
    const int j = threadIdx.x >> 4;  // row of the tile
    float* stage = stage_lds + (threadIdx.x >> 6) * stage_wave_words<E>();
    // its latest own tile; the grid's workgroups sweep the tiles side by side
    // (a ticket counter instead, an atomic per tile on one address, held the
    // whole chip to 47 tiles a microsecond: 86 us for 256 x N=65536)
    int own = first + (int)blockIdx.x;
    int tile = own, kind = kFusedOwn;
    // thread 0: the workgroup's listed tiles, those taken up again in vain,
    // a tile to help with, and the tasks taken beyond its own tiles
    int head = -1, again = -1, missing = -1, tries = 0;
    while (tile >= 0 && tile < total) {  // uniform
        const int q = tile >> lg_bps;
        const int ti = tile & (bps - 1);
        float* rows = loc.Rows(q);
        float* words = rows + 8 * (size_t)ti;
        const size_t lo = (size_t)ti * kFusedTile + (size_t)threadIdx.x * E;
        const size_t run = lo - (size_t)lane * E;
        RawPart<E> raw;
        float xo[E];
        unsigned long long seen = ~0ull;
        load_slices<E, HAS_B, CT>(loc, q, lo, run, stage, raw);
        if constexpr (REFINE) {
            // No tile stores x before every tile of its system is published,
            // so x as loaded here is the iterate's if this tile (for the
            // values inside it) or the tile beside it (for the value next to
            // it) is not published after the loads; else a helper was
            // quicker, and the tile beside it published the value.
            load_e<E>(loc.X(q) + lo, xo);
            float xl, xr;
            wave_halo<E>(loc.X(q), lo, loc.n, lane, xo, xl, xr);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads are complete before the reads below
            if (lane == 0) seen = read_pair(words);
            if (kind != kFusedOwn) {
                if (threadIdx.x == 0 && ti > 0) {
                    const unsigned long long v = read_pair(words - 2);
                    if (!pair_missing(v)) xl = pair_second(v);
                }
                if (threadIdx.x == kFusedThreads - 1 && ti + 1 < bps) {
                    const unsigned long long v = read_pair(words + 14);
                    if (!pair_missing(v)) xr = pair_first(v);
                }
            }
            residual_fp64<E, HAS_B>(xo, xl, xr, raw);
        }
        Fast16State<E> fs;
        fast16_stage1<E>(raw, HAS_B, l, fs);
        if (l == 0) {
            s_ends[0][j] = fs.sA;
            s_ends[1][j] = fs.sC;
            s_ends[2][j] = fs.sR;
        }
        if (l == 15) {
            s_ends[3][j] = fs.eA;
            s_ends[4][j] = fs.eC;
            s_ends[5][j] = fs.eR;
        }
        if constexpr (REFINE) {
            if (lane == 0) s_seen[threadIdx.x >> 6] = pair_missing(seen) ? 0 : 1;
            if (threadIdx.x == kFusedThreads - 1) s_xlast = xo[E - 1];
        }
        __syncthreads();
        if constexpr (REFINE) {
            if (kind != kFusedAgain && __builtin_amdgcn_readfirstlane(s_seen[0] | s_seen[1] | s_seen[2] | s_seen[3]) != 0) {
                // published by a helper before it was loaded: its own tile is
                // loaded again for the published x, another's is done with
                __syncthreads();
                if (kind == kFusedOwn) {
                    kind = kFusedAgain;
                    continue;
                }
            }
        }
        Chain16 ch;  // in every DPP row: lane l takes row l of the tile
        ch.reduce(BlockEnds{s_ends[0][l], s_ends[1][l], s_ends[2][l], s_ends[3][l], s_ends[4][l], s_ends[5][l]}, l);
        if (threadIdx.x < 64) {
            const bool skip = REFINE && kind == kFusedHelp && (s_seen[0] | s_seen[1] | s_seen[2] | s_seen[3]) != 0;
            const BlockEnds mine = ch.ends(0);
            if (threadIdx.x == 0 && kind != kFusedAgain && !skip) {
                if constexpr (REFINE) publish_pair(words + 6, xo[0], s_xlast);
                publish_ends(words, mine);
            }
            BlockEnds e{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            float before = 0.0f, after = 0.0f;
            unsigned long long m;  // lanes whose block is missing
            const int limit = kind == kFusedHelp ? 0 : spin;
            if constexpr (!WIDE) {
                m = wait_ends(rows + 8 * (size_t)lane, lane < bps, limit, e);
                if (m == 0) solve_blocks(e, bps, ti, lane, before, after);
                else missing = tile - ti + __builtin_ctzll(m);
            } else {
                const int g = ti / kFusedGroup, ng = bps / kFusedGroup;
                m = wait_ends(rows + 8 * (size_t)(g * kFusedGroup + l), lane < kFusedGroup, limit, e);
                if (m != 0) {
                    missing = tile - ti + g * kFusedGroup + __builtin_ctzll(m);
                } else {
                    Chain16 cg;
                    cg.reduce(e, l);
                    // every tile of the group publishes its equations (the
                    // same words), so that none waits for a particular one
                    const BlockEnds ge = cg.ends(0);
                    if (threadIdx.x == 0) publish_ends(fused_groups(rows, bps) + 8 * g, ge);
                    e = BlockEnds{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                    m = wait_ends(fused_groups(rows, bps) + 8 * lane, lane < ng, limit, e);
                    if (m != 0) {
                        missing = tile - ti + __builtin_ctzll(m) * kFusedGroup + tries % kFusedGroup;
                    } else {
                        float ob, oa, xb, xe, xa;
                        solve_blocks(e, ng, g, lane, ob, oa);
                        cg.solve(ob, oa, l, xb, xe, xa);
                        before = __shfl(xb, ti % kFusedGroup, 64);
                        after = __shfl(xa, ti % kFusedGroup, 64);
                    }
                }
            }
            if (threadIdx.x == 0) {
                s_side[0] = before;
                s_side[1] = after;
                s_ok = m == 0 ? 1 : 0;
            }
        }
        __syncthreads();
        const bool ok = __builtin_amdgcn_readfirstlane(s_ok) != 0;
        if (ok && kind != kFusedHelp) {
            float xb, xe, xa;
            ch.solve(s_side[0], s_side[1], l, xb, xe, xa);
            const int src = (lane & 48) + j;  // a lane that holds row j
            float X[E];
            fast16_finish<E>(fs, __shfl(xb, src, 64), __shfl(xe, src, 64), __shfl(xa, src, 64), l, X);
            if constexpr (REFINE) {
#pragma unroll
                for (int i = 0; i < E; i++) X[i] = xo[i] + X[i];
            }
            store_x_staged<E, true>(loc.X(q), X, stage, run, (size_t)loc.n, lane);
        }
        if (tile == own && own + stride < total && ok) {
            own += stride;
            tile = own;
            kind = kFusedOwn;
            continue;
        }
        // a tile to list, or no tile of its own left
        if (threadIdx.x == 0) {
            if (!ok && kind != kFusedHelp) {
                int& to = kind == kFusedOwn ? head : again;
                *fused_link(rows, bps, ti) = to;
                to = tile;
            }
            int t = -1, k = kFusedAgain;
            if (own + stride < total) {
                t = own + stride;
                k = kFusedOwn;
            } else if (tries < kFusedTries) {
                if (!ok && kind == kFusedAgain) {
                    t = missing;
                    k = kFusedHelp;
                } else {
                    if (head < 0) {
                        head = again;
                        again = -1;
                    }
                    if (head >= 0) {
                        t = head;
                        head = *fused_link(loc.Rows(t >> lg_bps), bps, t & (bps - 1));
                    }
                }
                tries++;
            }
            s_tile = t;
            s_kind = k;
        }
        __syncthreads();
        tile = __builtin_amdgcn_readfirstlane(s_tile);
        kind = __builtin_amdgcn_readfirstlane(s_kind);
        if (kind == kFusedOwn) own = tile;
    }
}

// Workgroups of `kernel` a device holds at once, with `lds` bytes of dynamic
// LDS each (0 on a query error).
template <typename K>
int resident_workgroups(K kernel, int threads, size_t lds) {
    int dev = 0, cus = 0, occ = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, threads, lds) != hipSuccess) return 0;
    return cus * occ;
}

template <bool HAS_B, typename CT, bool REFINE, bool WIDE, typename Loc>
hipError_t launch_fused_t(const Loc& loc, int n, int nsys, hipStream_t stream, bool* done) {
    const int lg_bps = __builtin_ctz((unsigned)(n / kFusedTile));
    const auto kern = fused_split_kernel<HAS_B, CT, REFINE, WIDE, Loc>;
    // workgroups resident at once, asked once per device: the query costs
    // the host as much as a launch
    static std::atomic<int> known[64];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    int capacity = dev < 64 ? known[dev].load(std::memory_order_relaxed) : 0;
    if (capacity == 0) {
        // a multiple of the group, so that a system's tiles run side by side
        // in every sweep of the grid over the tiles
        capacity = resident_workgroups(kern, kFusedThreads, 0) & ~(kFusedGroup - 1);
        if (dev < 64) known[dev].store(capacity, std::memory_order_relaxed);
    }
    *done = capacity >= 1 << lg_bps;
    if (!*done) return hipSuccess;
    const int tiles = nsys << lg_bps;
    const int grid = tiles < capacity ? tiles : capacity;
    hipLaunchKernelGGL((clear_fused_kernel<Loc>), dim3((tiles + 255) / 256), dim3(256), 0, stream, loc, nsys, lg_bps);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kFusedThreads), 0, stream, loc, nsys, lg_bps, 0, grid, kFusedSpin);
    return hipGetLastError();
}

// One round: nsys systems of n equations (n / kFusedTile tiles each) at loc.
// *done is false, and nothing is launched, where the device does not hold a
// whole system's workgroups at once (a refinement step on 4 Mi equations, at
// three workgroups per CU): every tile would be loaded twice (4 Mi equations:
// 104 us that way, 97 in two passes).
template <bool HAS_B, typename CT, bool REFINE, typename Loc>
hipError_t launch_fused(const Loc& loc, int n, int nsys, hipStream_t stream, bool* done) {
    return n / kFusedTile > kFusedWave ? launch_fused_t<HAS_B, CT, REFINE, true>(loc, n, nsys, stream, done)
                                       : launch_fused_t<HAS_B, CT, REFINE, false>(loc, n, nsys, stream, done);
}

}  // namespace tprh
