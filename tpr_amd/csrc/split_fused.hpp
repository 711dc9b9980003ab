// split_fused.hpp -- fast PTPR and TPR on systems larger than one workgroup in
// one pass: every equation is read once and x written once (20 B/eq), against
// 36 B/eq for the two passes of split_kernels.hpp.
//
// What bounds it: HBM.  The two passes move 604 MB for 256 x N=65536 at the
// rate such bytes can be moved (K1 46, K2 6, K3 47 us); reading the inputs
// once leaves 336 MB.  A whole solve of that batch: 101 us two passes, 63.5
// us this way (5.3 TB/s; a device copy of that size reaches 4.8-5.4); with an
// fp16-stored solve and a refinement step 203 -> 127.5 us; one system of 1 Mi
// equations 29.4 -> 11.4 us.
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
//   4. solves the system of the tiles' ends by the same steps (one tile per
//      lane) and finishes its rows from the unknowns on either side
//      of the tile (src/ptpr.cpp:263-287, x[ed+1] from the next row's first
//      equation instead of a division by c_ed).
// So one exchange of 24 bytes per 4096 equations crosses the chip, and the
// only wait is for the slowest tile of the system.  It needs no fence and no
// counter: the words are device-coherent, set to a NaN pattern that is never
// published before the launch (clear_fused_kernel), and a reader polls until
// no word of that pattern is left.  Four workgroups live on a CU at once, so
// that one's wait (4.1 us of a tile's 11 at the median) is covered by others'
// loads.
//
// Slices: s = 256 (one row), 512, 1024 or 2048 (several rows) -- in fast
// arithmetic a slice's interior, and the rows of a tile, may be eliminated in
// any order.  TPR runs its tree stages on every row instead of the two-level
// form, everything else alike (256 x N=65536, one
// buffer set: 100 us two passes, 58 us).
//
// The solve ends whichever workgroups are resident (fused_walk.hpp).
// Workgroup k of a grid of G takes tiles k, k + G, ...; it publishes a tile
// before it waits, and waits only `spin` polls: then it puts the tile on a
// list (linked through the workspace) and goes on with its next one.  Its own
// tiles done, it takes the listed ones up again (loading them again); where
// one still misses a tile, that tile's workgroup may not have started, and it
// computes and publishes the system's missing tiles, one after the other, on
// their workgroups' behalf (the same words), so each workgroup can finish
// with no other's help.  With a grid that the device holds at once, as
// launched here, on an otherwise idle device, no tile is ever listed.  The
// tasks that a workgroup can need have a bound (fused_task_limit), which only
// solves that overlap in one workspace, against its rule, could reach: a tile
// is then answered with NaN.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

#include "fused_walk.hpp"
#include "split_kernels.hpp"

namespace tprh {

constexpr int kFusedTile = 4096;               // equations per workgroup
constexpr int kFusedThreads = 256;
constexpr unsigned kFusedEmpty = 0xffffffffu;  // a word not yet published
constexpr int kFusedSpin = 64;                 // polls (about a microsecond each) before a tile is listed

// What the workgroups of one system exchange, in its boundary buffer (Rows)
// of bps tiles.  For block t (a tile; behind them a group of 16 tiles), its
// equations [F.a, F.c, F.r, L.a, L.c, L.r] (F: first unknown, L: last) are
// four words at ends4(t) and two at ends2(t), so that a wavefront reads 16
// blocks' words as three 128-byte lines: reads of one line from all over the
// chip are served one after the other, and polls are most of them.  x2: the
// iterate's x at a tile's ends (refinement); result: x just before and after
// a tile, found by its group's first; link: the list.  11 3/8 words per tile
// in all; the buffer has 8 per slice, two slices or more per tile.
struct FusedWords {
    float* rows;
    int bps;
    __device__ __forceinline__ int groups() const { return bps / kFusedGroup; }
    __device__ __forceinline__ float* ends4(int t) const { return rows + 4 * (size_t)t; }
    __device__ __forceinline__ float* ends2(int t) const { return rows + 4 * (size_t)bps + 2 * (size_t)t; }
    __device__ __forceinline__ float* x2(int t) const { return rows + 6 * (size_t)bps + 2 * (size_t)t; }
    __device__ __forceinline__ float* result(int t) const { return rows + 8 * (size_t)bps + 2 * (size_t)t; }
    __device__ __forceinline__ int* link(int t) const { return reinterpret_cast<int*>(rows) + 10 * (size_t)bps + t; }
    __device__ __forceinline__ float* group4(int g) const { return rows + 11 * (size_t)bps + 4 * g; }
    __device__ __forceinline__ float* group2(int g) const {
        return rows + 11 * (size_t)bps + 4 * (size_t)groups() + 2 * g;
    }
};

// Marks every published word empty (a kernel, not a memset, so that a
// captured graph replays it): the 10 words per tile ahead of the list links
// and the groups' behind them, in 16-byte pieces, one per thread.
__host__ __device__ inline int fused_clear_pieces(int bps) {
    return (10 * bps + (bps > kFusedGroup ? 6 * (bps / kFusedGroup) : 0)) / 4;
}
template <typename Loc>
__global__ __launch_bounds__(256) void clear_fused_kernel(Loc loc, int nsys, int bps) {
    const int pieces = fused_clear_pieces(bps);
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)nsys * pieces) return;
    const int q = (int)(i / pieces);
    int k = (int)(i - (long long)q * pieces);
    if (4 * k >= 10 * bps) k += bps / 4;  // the list links are not cleared
    reinterpret_cast<uint4*>(loc.Rows(q))[k] = make_uint4(kFusedEmpty, kFusedEmpty, kFusedEmpty, kFusedEmpty);
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

__device__ __forceinline__ void publish_ends(float* p4, float* p2, const BlockEnds& e) {
    publish_pair(p4, e.fa, e.fc);
    publish_pair(p4 + 2, e.fr, e.la);
    publish_pair(p2, e.lc, e.lr);
}
// False while a word is missing.  Two device-coherent loads (every word is
// checked by itself, so nothing wider than a word need be atomic).
__device__ __forceinline__ bool read_ends(const float* p4, const float* p2, BlockEnds& e) {
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    v4u a;
    v2u b;
    asm volatile("global_load_dwordx4 %0, %2, off sc1\n\t"
                 "global_load_dwordx2 %1, %3, off sc1\n\t"
                 "s_waitcnt vmcnt(0)"
                 : "=&v"(a), "=&v"(b)
                 : "v"(p4), "v"(p2)
                 : "memory");
    auto f = [](unsigned v) { return __builtin_bit_cast(float, v); };
    e = BlockEnds{f(a.x), f(a.y), f(a.z), f(a.w), f(b.x), f(b.y)};
    return a.x != kFusedEmpty && a.y != kFusedEmpty && a.z != kFusedEmpty && a.w != kFusedEmpty &&
           b.x != kFusedEmpty && b.y != kFusedEmpty;
}

// Polls until lanes with `need` have read their blocks' words into their e;
// after `limit` polls gives up.  Returns the lanes still missing theirs.
// Every lane of the wavefront calls this.
__device__ __forceinline__ unsigned long long wait_ends(const float* p4, const float* p2, bool need, int limit,
                                                        BlockEnds& e) {
    for (int i = 0;; i++) {
        if (need) need = !read_ends(p4, p2, e);
        const unsigned long long missing = __ballot(need);
        if (missing == 0 || i >= limit) return missing;
        __builtin_amdgcn_s_sleep(2);
    }
}
// The same for one published pair, in lane 0.
__device__ __forceinline__ unsigned long long wait_pair(const float* p, int lane, int limit, float& x, float& y) {
    unsigned long long v = 0, missing;
    bool need = lane == 0;
    for (int i = 0;; i++) {
        if (need) {
            v = read_pair(p);
            need = pair_missing(v);
        }
        missing = __ballot(need);
        if (missing == 0 || i >= limit) break;
        __builtin_amdgcn_s_sleep(2);
    }
    x = pair_first(v);
    y = pair_second(v);
    return missing;
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

// A whole system of up to 16 blocks, with ROWS up to 64, one per lane (lanes
// past the last one hold zero equations): x just before and just after block
// k (uniform).
template <bool ROWS>
__device__ __forceinline__ void solve_blocks(const BlockEnds& e, int count, int k, int lane, float& before,
                                             float& after) {
    const int l = lane & 15;
    Chain16 c;
    c.reduce(e, l);
    float ob = 0.0f, oa = 0.0f;  // x outside the lane's row
    if (ROWS && count > 16) {
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

// One lane's equations between the two halves of a row's solve: stage 1 into
// the row's ends (sA, sC, sR in lane 0; eA, eC, eR in lane 15), and x from
// the unknowns around the row once they are known.
template <int METHOD, int E>
struct RowState;
template <int E>
struct RowState<0, E> {  // PTPR: the two-level stage 1
    Fast16State<E> st;
    __device__ __forceinline__ void reduce(const RawPart<E>& raw, bool has_b, int l, BlockEnds& e) {
        fast16_stage1<E>(raw, has_b, l, st);
        e = BlockEnds{st.sA, st.sC, st.sR, st.eA, st.eC, st.eR};
    }
    __device__ __forceinline__ void finish(float before, float last, float after, int l, float (&X)[E]) const {
        fast16_finish<E>(st, before, last, after, l, X);
    }
};
template <int E>
struct RowState<1, E> {  // TPR: the tree (src/tpr.cpp:123-230, :277-308)
    float A[E], C[E], R[E], Ao[E], Co[E], Ro[E];
    __device__ __forceinline__ void reduce(const RawPart<E>& raw, bool has_b, int l, BlockEnds& e) {
        normalise<E, kFast>(raw, has_b, A, C, R);
#pragma unroll
        for (int i = 0; i < E; i++) {
            Ao[i] = A[i];
            Co[i] = C[i];
            Ro[i] = R[i];
        }
        tpr_stage1_level<E, 16, kFast, 1>(A, C, R, l);
        e = BlockEnds{A[0], C[0], R[0], A[E - 1], C[E - 1], R[E - 1]};
    }
    __device__ __forceinline__ void finish(float before, float last, float, int l, float (&X)[E]) const {
        tpr_stage3<E, 16, kFast>(A, C, R, Ao, Co, Ro, before, last, l, X);
    }
};

// What a wavefront reads and publishes of a system of groups (fused_look).
struct GroupWords {
    const FusedWords fw;
    const int lane;
    BlockEnds e;  // of the blocks last read, one per lane; past the last one zero equations

    __device__ __forceinline__ unsigned long long tiles(int g, int limit) {
        const int t = g * kFusedGroup + (lane & 15);
        e = BlockEnds{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        return wait_ends(fw.ends4(t), fw.ends2(t), lane < kFusedGroup, limit, e);
    }
    __device__ __forceinline__ unsigned long long groups(int limit) {
        e = BlockEnds{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        return wait_ends(fw.group4(lane), fw.group2(lane), lane < fw.groups(), limit, e);
    }
    __device__ __forceinline__ Chain16 publish(int g) {
        Chain16 c;
        c.reduce(e, lane & 15);
        const BlockEnds ge = c.ends(0);
        if (lane == 0) publish_ends(fw.group4(g), fw.group2(g), ge);
        return c;
    }
};

// WIDE: more than 16 tiles per system (up to 1024): the exchange goes through
// groups of 16 tiles -- the group's first tile reduces it, exchanges its ends
// with the other groups', and hands every tile of the group the x on its
// sides -- so that a tile polls one word pair and no line is polled by more
// than 64 workgroups.  Reads of one line from all over the chip are served
// one after the other: with every tile polling every group's words, 16
// systems of 1 Mi equations took 237 us, this way 78; with every tile polling
// all of up to 64 tiles' words, 64 systems of 256 Ki 73 us, this way 59.
template <int METHOD, bool HAS_B, typename CT, bool REFINE, bool WIDE, typename Loc>
__global__ __launch_bounds__(kFusedThreads, REFINE ? 3 : 4) void fused_split_kernel(Loc loc, int nsys, int lg_bps, int first,
                                                                                    int stride, int spin, int tasks) {
    constexpr int E = 16;
    __shared__ __align__(16) float stage_lds[stage_words<E>(kFusedThreads)];
    __shared__ float s_ends[6][16];  // E_st and E_ed of the tile's rows
    __shared__ float s_side[2];      // x just before and just after the tile
    __shared__ int s_seen[4];        // per wavefront: the tile was published before it was loaded
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
    FusedWalk walk;    // thread 0's
    int missing = -1;  // a tile to help with
    while (tile >= 0 && tile < total) {  // uniform
        const int q = tile >> lg_bps;
        const int ti = tile & (bps - 1);
        const FusedWords fw{loc.Rows(q), bps};
        const size_t lo = (size_t)ti * kFusedTile + (size_t)threadIdx.x * E;
        const size_t run = lo - (size_t)lane * E;
        RawPart<E> raw;
        float xo[E];
        unsigned long long seen = ~0ull;  // in lane 0
        float tile_end = 0.0f;            // refinement: the iterate's last x of the tile, in thread 0
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
            if (threadIdx.x == 0) tile_end = loc.X(q)[lo + kFusedTile - 1];
            // the loads are complete before the reads below (xl and xr: the
            // compiler would else wait for them, and so for all of those, where
            // the values are used)
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(xl), "+v"(xr), "+v"(tile_end)::"memory");
            // x at the tile's ends, for whoever loads a tile beside it later.
            // An own tile's x is the iterate's until this workgroup stores it
            if (threadIdx.x == 0 && kind == kFusedOwn) publish_pair(fw.x2(ti), xo[0], tile_end);
            if (lane == 0) seen = read_pair(fw.ends2(ti));
            if (kind != kFusedOwn) {
                if (threadIdx.x == 0 && ti > 0) {
                    const unsigned long long v = read_pair(fw.x2(ti - 1));
                    if (!pair_missing(v)) xl = pair_second(v);
                }
                if (threadIdx.x == kFusedThreads - 1 && ti + 1 < bps) {
                    const unsigned long long v = read_pair(fw.x2(ti + 1));
                    if (!pair_missing(v)) xr = pair_first(v);
                }
            }
            residual_fp64<E, HAS_B>(xo, xl, xr, raw);
        }
        RowState<METHOD, E> row;
        BlockEnds re;
        row.reduce(raw, HAS_B, l, re);
        if (l == 0) {
            s_ends[0][j] = re.fa;
            s_ends[1][j] = re.fc;
            s_ends[2][j] = re.fr;
        }
        if (l == 15) {
            s_ends[3][j] = re.la;
            s_ends[4][j] = re.lc;
            s_ends[5][j] = re.lr;
        }
        if constexpr (REFINE) {
            if (lane == 0) s_seen[threadIdx.x >> 6] = pair_missing(seen) ? 0 : 1;
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
            const BlockEnds mine = ch.ends(0);
            bool there_before = false;  // of a tile of another's: published when all its loads were complete
            if (threadIdx.x == 0 && kind == kFusedHelp) {
                if constexpr (REFINE) there_before = (s_seen[0] | s_seen[1] | s_seen[2] | s_seen[3]) != 0;
                else there_before = !pair_missing(read_pair(fw.ends2(ti)));
            }
            if (threadIdx.x == 0 && fused_publishes(kind, there_before)) {
                if constexpr (REFINE) {
                    // x2 is there before the tile's words are, and so before any
                    // x of the tile is stored
                    if (kind == kFusedHelp) publish_pair(fw.x2(ti), xo[0], tile_end);
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
                publish_ends(fw.ends4(ti), fw.ends2(ti), mine);
            }
            BlockEnds e{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            float before = 0.0f, after = 0.0f;
            bool there;  // every block that this tile waits for
            const int limit = kind == kFusedHelp ? 0 : spin;
            if constexpr (!WIDE) {
                const unsigned long long m = wait_ends(fw.ends4(lane), fw.ends2(lane), lane < bps, limit, e);
                there = m == 0;
                if (__builtin_expect(there, 1)) solve_blocks<false>(e, bps, ti, lane, before, after);
                else missing = tile - ti + fused_pick(m, ti);
            } else if (ti % kFusedGroup != 0 && kind == kFusedOwn) {
                there = wait_pair(fw.result(ti), lane, limit, before, after) == 0;
            } else {
                // the group's first tile reduces the group, solves the system
                // of the groups and hands every tile of the group its sides
                // (a tile taken up again does so by itself)
                const int g = ti / kFusedGroup;
                GroupWords gw{fw, lane};
                int lost = -1;
                if (__builtin_expect(kind != kFusedOwn, 0)) lost = fused_look(gw, ti, limit);
                there = lost < 0 && gw.tiles(g, limit) == 0;
                if (there) {
                    const Chain16 chain = gw.publish(g);
                    there = gw.groups(limit) == 0;
                    if (there) {
                        float ob, oa, xb, xe, xa;
                        solve_blocks<true>(gw.e, fw.groups(), g, lane, ob, oa);
                        chain.solve(ob, oa, l, xb, xe, xa);
                        if (lane < kFusedGroup) publish_pair(fw.result(g * kFusedGroup + l), xb, xa);
                        before = __shfl(xb, ti % kFusedGroup, 64);
                        after = __shfl(xa, ti % kFusedGroup, 64);
                    }
                }
                missing = tile - ti + lost;
            }
            if (threadIdx.x == 0) {
                const bool lost = !there && kind == kFusedAgain && walk.lost(tasks);  // its x: NaN
                s_side[0] = lost ? __builtin_nanf("") : before;
                s_side[1] = lost ? __builtin_nanf("") : after;
                s_ok = there || lost ? 1 : 0;
            }
        }
        __syncthreads();
        const bool ok = __builtin_amdgcn_readfirstlane(s_ok) != 0;
        if (__builtin_expect(ok && kind != kFusedHelp, 1)) {
            float xb, xe, xa;
            ch.solve(s_side[0], s_side[1], l, xb, xe, xa);
            const int src = (lane & 48) + j;  // a lane that holds row j
            float X[E];
            row.finish(__shfl(xb, src, 64), __shfl(xe, src, 64), __shfl(xa, src, 64), l, X);
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
            const FusedTask t = walk.next(tile, kind, ok, missing, own + stride < total ? own + stride : -1, tasks,
                                          [&](int k) -> int& {
                                              return *FusedWords{loc.Rows(k >> lg_bps), bps}.link(k & (bps - 1));
                                          });
            s_tile = t.tile;
            s_kind = t.kind;
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

// CUs that a stream's kernels run on, of the device's `cus`: fewer on a stream
// made with a CU mask (0.3 us on the host).  The mask query takes neither the
// null stream's legacy handle nor a stream destroyed, which the launch refuses.
inline int stream_cus(hipStream_t stream, int cus) {
    uint32_t mask[32] = {};
    hipDevice_t dev;
    if (stream == hipStreamLegacy) stream = nullptr;
    if ((stream && hipStreamGetDevice(stream, &dev) != hipSuccess) ||
        hipExtStreamGetCUMask(stream, 32, mask) != hipSuccess) {
        (void)hipGetLastError();
        return cus;
    }
    int n = 0;
    for (uint32_t w : mask) n += __builtin_popcount(w);
    return n > 0 && n < cus ? n : cus;
}

template <int METHOD, bool HAS_B, typename CT, bool REFINE, bool WIDE, typename Loc>
hipError_t launch_fused_t(const Loc& loc, int n, int nsys, hipStream_t stream, bool* done) {
    const int lg_bps = __builtin_ctz((unsigned)(n / kFusedTile));
    const auto kern = fused_split_kernel<METHOD, HAS_B, CT, REFINE, WIDE, Loc>;
    // workgroups resident at once: those of a CU and the CUs, asked once per
    // device (the query costs the host as much as a launch), times the
    // stream's share of the CUs
    static std::atomic<int> known_cus[64], known_all[64];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    int cus = dev < 64 ? known_cus[dev].load(std::memory_order_acquire) : 0;
    int all = cus ? known_all[dev].load(std::memory_order_relaxed) : 0;
    if (cus == 0) {
        all = resident_workgroups(kern, kFusedThreads, 0);
        if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
        if (dev < 64) {
            known_all[dev].store(all, std::memory_order_relaxed);
            known_cus[dev].store(cus, std::memory_order_release);
        }
    }
    // a multiple of the group, so that a system's tiles run side by side in
    // every sweep of the grid over the tiles
    const int capacity = (int)((long long)all * stream_cus(stream, cus) / cus) & ~(kFusedGroup - 1);
    *done = capacity >= 1 << lg_bps;
    if (!*done) return hipSuccess;
    const int tiles = nsys << lg_bps;
    const int grid = tiles < capacity ? tiles : capacity;
    const long long pieces = (long long)nsys * fused_clear_pieces(1 << lg_bps);
    hipLaunchKernelGGL((clear_fused_kernel<Loc>), dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream, loc,
                       nsys, 1 << lg_bps);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kFusedThreads), 0, stream, loc, nsys, lg_bps, 0, grid, kFusedSpin,
                       fused_task_limit(tiles, grid, 1 << lg_bps));
    return hipGetLastError();
}

// One round: nsys systems of n equations (n / kFusedTile tiles each) at loc.
// *done is false, and nothing is launched, where the stream's CUs do not hold
// a whole system's workgroups at once (a refinement step on 4 Mi equations, at
// three workgroups per CU; a stream with a CU mask): every tile would be
// loaded twice or more (4 Mi equations: 104 us that way, 97 in two passes; 1
// Mi on 32 CUs 478, 87).
template <int METHOD, bool HAS_B, typename CT, bool REFINE, typename Loc>
hipError_t launch_fused(const Loc& loc, int n, int nsys, hipStream_t stream, bool* done) {
    return n / kFusedTile > kFusedGroup ? launch_fused_t<METHOD, HAS_B, CT, REFINE, true>(loc, n, nsys, stream, done)
                                       : launch_fused_t<METHOD, HAS_B, CT, REFINE, false>(loc, n, nsys, stream, done);
}

}  // namespace tprh
