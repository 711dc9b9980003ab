// solve_slot.hpp -- one system solved by one group of lanes of a workgroup,
// from per-system offsets.  Shared by the kernels (uneven batches, serving
// batches) that put systems of different sizes and layouts into one launch.
//
// In workgroups of kSlotTile lanes, slices of 8 and 16 equations per lane are
// read and written as staged_io.hpp does, 16-byte pieces in the order of
// memory turned through LDS.  A wavefront's 64 lanes may hold several systems
// (n / E < 64 lanes each) that lie anywhere; a piece then takes its address
// from the lane it belongs to.  In workgroups of 1024 lanes, of which a CU
// holds one, nothing covers the turn, and 20000 systems of 256 to 16384 took
// 545 us in place of 388: there each lane loads its own run.
// Exact PTPR runs its levels inside the lane in both (exact_rows.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include "launch_uneven.hpp"
#include "slice_solvers.hpp"
#include "staged_io.hpp"

namespace tprh {

// A ticket of a persistent kernel, read when it is used: to the compiler the
// address differs between lanes, or it adds the wavefront's lanes up first and
// waits for the counter's answer right here.
__device__ __forceinline__ int next_ticket(int* counter) {
    int zero = 0;
    asm volatile("" : "+v"(zero));
    return atomicAdd(counter + zero, 1);
}

// Where a lane's equations lie: floats from the bases of the coefficients,
// the right-hand sides and the answers to the lane's first equation.
struct SlotAt {
    size_t coef, rhs, x;
};

// Offset of the wavefront's 16-byte piece q, given every lane's own offset
// (its E / 4 pieces from there on).  Every lane of the wavefront calls this.
template <int E>
__device__ __forceinline__ size_t slot_piece(size_t own, int lg_lanes, int q) {
    if (lg_lanes >= 6) {  // one system: one run from lane 0 on
        const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)own);
        const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(own >> 32));
        return (((size_t)hi << 32) | lo) + 4 * (size_t)q;
    }
    const int from = q / (E / 4);
    const unsigned lo = __shfl((unsigned)own, from);
    const unsigned hi = __shfl((unsigned)(own >> 32), from);
    return (((size_t)hi << 32) | lo) + 4 * (size_t)(q % (E / 4));
}

// The workgroup's BLOCK lanes are cut into groups of 2^lg_lanes = m * L lanes, one
// system each (slot = threadIdx.x >> lg_lanes), of n = m * E * L equations;
// at: the lane's place in a / b / c, d and x.  Slots from `count` on have no
// system of their own: their offsets name another, they compute but never
// store.  lds: slot_lds_bytes of it.  Every lane of the workgroup must call this (the
// reduced solve has workgroup barriers); m, lg_lanes and count are uniform
// across the workgroup.
template <int METHOD, int MODE, bool HAS_B, int E, int L, int BLOCK>
__device__ __forceinline__ void solve_slot(int m, int lg_lanes, int count, const float* __restrict__ a,
                                           const float* __restrict__ b, const float* __restrict__ c,
                                           const float* __restrict__ d, float* __restrict__ x, const SlotAt& at,
                                           float* lds) {
    constexpr bool STAGE = kStageX<E> && BLOCK == kSlotTile;
    constexpr bool TURN = METHOD == 0 && MODE == kExact && kExactTurn<E, L>;
    // not known to be the same in every item, or the LDS addresses of every
    // shape are computed ahead of the kernel's loop and held: 172 bytes of
    // spills per lane
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int slot = tid >> lg_lanes;
    const int t = tid & ((1 << lg_lanes) - 1);
    const int lane = tid & 63;
    float* stage = lds + slot_row_words(BLOCK) + (tid >> 6) * stage_wave_words<E>();
    RawPart<E> raw;
    if constexpr (STAGE) {
        stage_v4f la[E / 4], lb[E / 4], lc[E / 4], ld[E / 4];
#pragma unroll
        for (int k = 0; k < E / 4; k++) {
            const size_t g = slot_piece<E>(at.coef, lg_lanes, k * 64 + lane);
            la[k] = *reinterpret_cast<const stage_v4f*>(a + g);
            lc[k] = *reinterpret_cast<const stage_v4f*>(c + g);
            if constexpr (HAS_B) lb[k] = *reinterpret_cast<const stage_v4f*>(b + g);
        }
#pragma unroll
        for (int k = 0; k < E / 4; k++)
            ld[k] = *reinterpret_cast<const stage_v4f*>(d + slot_piece<E>(at.rhs, lg_lanes, k * 64 + lane));
        turn_run<E>(la, stage, lane, raw.a, a);
        turn_run<E>(lc, stage, lane, raw.c, a);
        if constexpr (HAS_B) turn_run<E>(lb, stage, lane, raw.b, a);
        turn_run<E>(ld, stage, lane, raw.d, d);
    } else {
        // one array after the other: a lane's 64 bytes of one are a line that
        // the first 16 fetch; with the arrays' pieces in turn that line is
        // gone from the L1 before the others (20000 systems of 256 to 16384:
        // 388 -> 458 us)
        load_e<E>(a + at.coef, raw.a);
        __builtin_amdgcn_sched_barrier(0);
        load_e<E>(c + at.coef, raw.c);
        __builtin_amdgcn_sched_barrier(0);
        load_e<E>(d + at.rhs, raw.d);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (HAS_B) load_e<E>(b + at.coef, raw.b);
        __builtin_amdgcn_sched_barrier(0);
    }
    float X[E];
    float* my = lds + slot * lds_words_per_system(m);
    if constexpr (METHOD == 0) {
        ptpr_solve_raw<E, L, MODE, false, TURN>(raw, HAS_B, m, t, my, X, stage, lane);
    } else {
        float A[E], C[E], R[E];
        normalise<E, MODE>(raw, HAS_B, A, C, R);
        tpr_solve_regs<E, L, MODE>(A, C, R, m, t, my, X);
    }
    if constexpr (STAGE) {
        size_t own = at.x;
        asm volatile("" : "+v"(own));  // or the loads' addresses stay in registers until here
        stage_v4f* s4 = reinterpret_cast<stage_v4f*>(stage);
#pragma unroll
        for (int i = 0; i < E / 4; i++)
            s4[stage_slot(lane * (E / 4) + i)] = stage_v4f{X[4 * i], X[4 * i + 1], X[4 * i + 2], X[4 * i + 3]};
        group_sync<true>();
#pragma unroll
        for (int k = 0; k < E / 4; k++) {
            const int q = k * 64 + lane;
            const size_t g = slot_piece<E>(own, lg_lanes, q);
            const stage_v4f v = s4[stage_slot(q)];
            if ((int)((tid - lane + q / (E / 4)) >> lg_lanes) < count)
                *reinterpret_cast<stage_v4f*>(x + g) = v;
        }
        group_sync<true>();
    } else {
        if (slot < count) store_e<E>(x + at.x, X);
    }
}

}  // namespace tprh
