// staged_io.hpp -- a wavefront's loads and stores of 64 lanes x E
// consecutive floats as 1 KB runs per instruction.
//
// Every kernel here gives lane t of a system the equations [t E, t E + E),
// so the 64 lanes of a wavefront own one contiguous run of 64 E floats of
// each array.  Accessed lane by lane, each 16-byte load or store instruction
// touches a quarter (E = 16) of 64 separate 64-byte pieces; the non-temporal
// stores then reach memory as partial lines (WRITE_SIZE 1.5 times the bytes
// of x on 4096 x N=1024).  Passed through 68 E floats of LDS per wavefront,
// every instruction covers 1 KB of consecutive bytes instead, whole lines:
// 4096 x N=1024 batched PTPR 18.6 -> 14.3-14.8 us.
#pragma once
#include <hip/hip_runtime.h>

#include "launch.hpp"
#include "slice_solvers.hpp"

namespace tprh {

// The shapes that stage (16-byte pieces of the lanes' runs).
template <int E>
constexpr bool kStageX = E == 8 || E == 16 || E == 32;

// The 16-byte pieces of a wavefront's run sit in LDS with one spare slot
// after every 16 (slot q + q / 16): the per-lane reads and writes of 4 or 2
// consecutive pieces, like the per-instruction ones of 64 consecutive
// pieces, then fall on 16 different 16-byte bank groups in every group of
// 16 lanes, free of bank conflicts.
__device__ __forceinline__ int stage_slot(int q) { return q + (q >> 4); }

// LDS words per wavefront, and per workgroup of `lanes` lanes, for the
// staging: 17 E / 16 slots of 16 bytes per lane.
template <int E>
__host__ __device__ constexpr int stage_wave_words() { return 68 * E; }
template <int E>
__host__ __device__ constexpr int stage_words(int lanes) { return (lanes / 64) * stage_wave_words<E>(); }

// Start of the staging area behind spb systems' rows of m slices (16-byte
// aligned).
__host__ __device__ constexpr int stage_base(int spb, int m) { return (spb * lds_words_per_system(m) + 3) & ~3; }

typedef float stage_v4f __attribute__((ext_vector_type(4)));

// stage: the wavefront's stage_wave_words<E>() floats of LDS.
// Stores X of the 64 lanes to x[run .. run + 64 E): the wavefront's run.
// Pieces at or past `total` are not stored (lanes of systems past the end of
// a batch).  Every lane of the wavefront calls this.  NT: non-temporal.
template <int E, bool NT>
__device__ __forceinline__ void store_x_staged(float* __restrict__ x, const float (&X)[E], float* stage, size_t run,
                                               size_t total, int lane) {
    stage_v4f* s4 = reinterpret_cast<stage_v4f*>(stage);
#pragma unroll
    for (int i = 0; i < E / 4; i++)
        s4[stage_slot(lane * (E / 4) + i)] = stage_v4f{X[4 * i], X[4 * i + 1], X[4 * i + 2], X[4 * i + 3]};
    group_sync<true>();
#pragma unroll
    for (int k = 0; k < E / 4; k++) {
        const int q = k * 64 + lane;  // 16-byte piece of the run
        const size_t gi = run + 4 * (size_t)q;
        const stage_v4f v = s4[stage_slot(q)];
        if (gi < total) {
            if constexpr (NT) __builtin_nontemporal_store(v, reinterpret_cast<stage_v4f*>(x + gi));
            else *reinterpret_cast<stage_v4f*>(x + gi) = v;
        }
    }
    group_sync<true>();  // the area may be written again
}

// The lane's E values of one array out of the 16-byte pieces that the
// wavefront loaded of it (piece k * 64 + lane in l[k]), turned through LDS:
// E / 4 pieces of floats, or E / 8 of fp16 values, widened (exact).
template <int E>
__device__ __forceinline__ void turn_run(const stage_v4f (&l)[E / 4], float* stage, int lane, float (&out)[E],
                                         const float*) {
    stage_v4f* s4 = reinterpret_cast<stage_v4f*>(stage);
#pragma unroll
    for (int k = 0; k < E / 4; k++) s4[stage_slot(k * 64 + lane)] = l[k];
    group_sync<true>();
#pragma unroll
    for (int i = 0; i < E / 4; i++) {
        const stage_v4f v = s4[stage_slot(lane * (E / 4) + i)];
        out[4 * i] = v.x;
        out[4 * i + 1] = v.y;
        out[4 * i + 2] = v.z;
        out[4 * i + 3] = v.w;
    }
    group_sync<true>();
}
template <int E>
__device__ __forceinline__ void turn_run(const stage_v4f (&l)[E / 8], float* stage, int lane, float (&out)[E],
                                         const _Float16*) {
    typedef _Float16 v8h __attribute__((ext_vector_type(8)));
    stage_v4f* s4 = reinterpret_cast<stage_v4f*>(stage);
    if constexpr (E > 8) {
#pragma unroll
        for (int k = 0; k < E / 8; k++) s4[stage_slot(k * 64 + lane)] = l[k];
        group_sync<true>();
    }
#pragma unroll
    for (int i = 0; i < E / 8; i++) {
        const stage_v4f w = E > 8 ? s4[stage_slot(lane * (E / 8) + i)] : l[0];
        const v8h v = __builtin_bit_cast(v8h, w);
#pragma unroll
        for (int k = 0; k < 8; k++) out[8 * i + k] = (float)v[k];
    }
    if constexpr (E > 8) group_sync<true>();
}

// Loads the lane's E values of a, b (HAS_B), c (float or fp16) and d from the
// wavefront's run at `run`, as 1 KB per instruction.  CLAMP: pieces at or
// past `total` load the last piece before it instead (lanes that never
// store); without it the whole run lies below `total`.  Every lane of the
// wavefront calls this.
template <int E, bool HAS_B, bool CLAMP = true, typename CT = float>
__device__ __forceinline__ void load_raw_staged(const CT* __restrict__ a, const CT* __restrict__ b,
                                                const CT* __restrict__ c, const float* __restrict__ d, size_t run,
                                                size_t total, float* stage, int lane, RawPart<E>& p) {
    constexpr int V = 16 / (int)sizeof(CT);  // values per piece
    constexpr int K = E / V;                 // pieces per lane
    // the lane's k-th piece of an array of v values per piece
    auto load = [&](const auto* q, int k, int v) {
        size_t g = run + (size_t)v * (size_t)(k * 64 + lane);
        if (CLAMP) g = g < total ? g : total - (size_t)v;
        return *reinterpret_cast<const stage_v4f*>(q + g);
    };
    stage_v4f la[K], lb[K], lc[K], ld[E / 4];
#pragma unroll
    for (int k = 0; k < K; k++) la[k] = load(a, k, V);
#pragma unroll
    for (int k = 0; k < K; k++) lc[k] = load(c, k, V);
#pragma unroll
    for (int k = 0; k < E / 4; k++) ld[k] = load(d, k, 4);
    if constexpr (HAS_B) {
#pragma unroll
        for (int k = 0; k < K; k++) lb[k] = load(b, k, V);
    }
    turn_run<E>(la, stage, lane, p.a, a);
    turn_run<E>(lc, stage, lane, p.c, a);
    turn_run<E>(ld, stage, lane, p.d, d);
    if constexpr (HAS_B) turn_run<E>(lb, stage, lane, p.b, a);
}

// x just before and just after the lane's E values xo: from the lanes beside
// it, at the wavefront's ends from memory (0 outside the system's [0, n)).
// lo: the lane's first equation in the system at x.
template <int E>
__device__ __forceinline__ void wave_halo(const float* __restrict__ x, size_t lo, int n, int lane,
                                          const float (&xo)[E], float& xl, float& xr) {
    xl = shift_up<64, 1>(xo[E - 1], 0.0f, lane);
    xr = shift_down<64, 1>(xo[0], 0.0f, lane);
    if (lane == 0 && lo > 0) xl = x[lo - 1];
    if (lane == 63 && lo + E < (size_t)n) xr = x[lo + E];
}

}  // namespace tprh
