// exact_rows.hpp -- PTPR stage 1 in exact arithmetic (src/ptpr.cpp:130-190)
// with most of its levels inside the lane.
//
// What bounds it: the vector ALU.  Bit identity leaves the reference's
// operations as they are: at each of log2 S levels every equation takes nine
// products, four sums and an IEEE reciprocal, none of them fused.  For
// 4096 x N=1024 the instructions left here take 21 us to issue (2450 and 170
// reciprocal seeds per wavefront, at 4 and 16 cycles; 18 with quots_rn), its
// memory traffic 14.
// So what can be saved is everything else: exchanges between lanes, selects
// for missing partners, and the guard and branch of each reciprocal.
//
// A slice of S = E L equations starts blocked, equation l E + e in register e
// of lane l: the levels u = 1 .. E/2 find their partners in the lane, but for
// u equations at each end.  After that the equations are turned through LDS
// (24 bytes each way per equation), equation e L + l in register e of lane l:
// the levels u = L .. S/2 find all partners in the lane, u / L registers away,
// and which are missing is known to the compiler.  Only the levels E <= u < L
// (none for E = L = 16) exchange whole registers between lanes.
//
// The off-diagonals are kept negated (Ap = -a, Cp = -c), which changes no
// rounding: in that form a missing partner is a product of +0 in the
// denominator, of -0 in the right-hand side (which may itself be -0, and
// -0 + +0 would be +0) and a factor 1 in the off-diagonal, so the upper and
// lower formulas (src/ptpr.cpp:140-152, :171-182) take no selects: the fused
// DPP products leave the lanes without a partner alone.
// A level's reciprocals share one range test and one wave-uniform branch.
//
// Measured (fp32 with a diagonal; the register form before -> this form ->
// with the quotients of quots_rn), 4096 systems of N = 1024: 16 x 16 42.5 ->
// 28.1 -> 25.4 us (8 x 32 39.2 -> 32.4, 4 x 64, which stays in registers,
// 34.8), 16 x 32 50.4 -> 31.2, 8 x 64 41.9 -> 34.2; 512 of N = 8192, S = 2048
// (32 x 64) 111 -> 38.5.  One system of N = 1024: 8 x 32 10.8 -> 7.1 -> 6.9,
// 4 x 64 7.0.  Exact TPR, which divides alike, 20.5 -> 18.6 on the 4096.
#pragma once
#include <hip/hip_runtime.h>

#include "tpr_device.hpp"

namespace tprh {

// Word w of a wavefront's 64 E values in its LDS area of 68 E floats: one
// spare 16-byte slot after every 16, as in staged_io.hpp, so that runs of
// consecutive words and runs of E words per lane are both free of bank
// conflicts.
__device__ __forceinline__ int turn_word(int w) { return w + 4 * (w >> 6); }

// v[e] = equation l E + e of the lane's slice  ->  v[e] = equation e L + l.
// Every lane of the wavefront calls this.
template <int E, int L>
__device__ __forceinline__ void turn_strided(float (&v)[E], float* area, int lane) {
    typedef float v4f __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < E / 4; i++)
        *reinterpret_cast<v4f*>(area + turn_word(lane * E + 4 * i)) =
            v4f{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
    group_sync<true>();
    const int base = (lane / L) * (E * L) + lane % L;
#pragma unroll
    for (int e = 0; e < E; e++) v[e] = area[turn_word(base + e * L)];
    group_sync<true>();
}
// And back.
template <int E, int L>
__device__ __forceinline__ void turn_blocked(float (&v)[E], float* area, int lane) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    const int base = (lane / L) * (E * L) + lane % L;
#pragma unroll
    for (int e = 0; e < E; e++) area[turn_word(base + e * L)] = v[e];
    group_sync<true>();
#pragma unroll
    for (int i = 0; i < E / 4; i++) {
        const v4f w = *reinterpret_cast<const v4f*>(area + turn_word(lane * E + 4 * i));
        v[4 * i] = w.x;
        v[4 * i + 1] = w.y;
        v[4 * i + 2] = w.z;
        v[4 * i + 3] = w.w;
    }
    group_sync<true>();
}

// p = s(lane - D) * m and q = t(lane - D) * m; +0 and -0 in the first D lanes
// of the slice.
template <int L, int D>
__device__ __forceinline__ void exact_mul_up(float s, float t, float m, int l, float& p, float& q) {
    p = 0.0f;
    q = -0.0f;
    if constexpr (L == 16) {
        asm("s_nop 1\n\t"
            "v_mul_f32_dpp %[p], %[s], %[m] row_shr:%[d] row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %[q], %[t], %[m] row_shr:%[d] row_mask:0xf bank_mask:0xf"
            : [p] "+&v"(p), [q] "+&v"(q)
            : [s] "v"(s), [t] "v"(t), [m] "v"(m), [d] "i"(D));
    } else {
        const float x = shift_up<L, D>(s, 0.0f, l) * m, y = shift_up<L, D>(t, 0.0f, l) * m;
        p = l >= D ? x : 0.0f;
        q = l >= D ? y : -0.0f;
    }
}
// The same from lane + D, +0 and -0 in the last D lanes.
template <int L, int D>
__device__ __forceinline__ void exact_mul_dn(float s, float t, float m, int l, float& p, float& q) {
    p = 0.0f;
    q = -0.0f;
    if constexpr (L == 16) {
        asm("s_nop 1\n\t"
            "v_mul_f32_dpp %[p], %[s], %[m] row_shl:%[d] row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %[q], %[t], %[m] row_shl:%[d] row_mask:0xf bank_mask:0xf"
            : [p] "+&v"(p), [q] "+&v"(q)
            : [s] "v"(s), [t] "v"(t), [m] "v"(m), [d] "i"(D));
    } else {
        const float x = shift_down<L, D>(s, 0.0f, l) * m, y = shift_down<L, D>(t, 0.0f, l) * m;
        p = l < L - D ? x : 0.0f;
        q = l < L - D ? y : -0.0f;
    }
}
// s(lane - D) * u, or u in the first D lanes; s(lane + D) * u, or u in the
// last D.
template <int L, int D>
__device__ __forceinline__ float exact_keep_up(float s, float u, int l) {
    if constexpr (L == 16) return dpp_keep_mul_up<D>(s, u);
    else {
        const float p = shift_up<L, D>(s, 1.0f, l) * u;
        return l >= D ? p : u;
    }
}
template <int L, int D>
__device__ __forceinline__ float exact_keep_dn(float s, float u, int l) {
    if constexpr (L == 16) return dpp_keep_mul_dn<D>(s, u);
    else {
        const float p = shift_down<L, D>(s, 1.0f, l) * u;
        return l < L - D ? p : u;
    }
}

// x[k] -> 1 / x[k], rounded as IEEE division does: the short sequence of
// recip_rn without its fixup, which equals division for every |x| in
// [2^-126, 2^126] and for NaN (checked on every float by
// tests/test_gpu_exact_rows.py), else division.  One branch for the
// wavefront.
__device__ __forceinline__ float recip_short(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}
template <int E>
__device__ __forceinline__ void recips_rn(float (&x)[E]) {
    float mn = __builtin_fabsf(x[0]), mx = mn;
#pragma unroll
    for (int k = 1; k < E; k++) {
        mn = __builtin_fminf(mn, __builtin_fabsf(x[k]));
        mx = __builtin_fmaxf(mx, __builtin_fabsf(x[k]));
    }
    const bool plain = mn >= 0x1p-126f && mx <= 0x1p126f;
    if (__ballot(!plain) == 0) {
#pragma unroll
        for (int k = 0; k < E; k++) x[k] = recip_short(x[k]);
    } else {
#pragma unroll
        for (int k = 0; k < E; k++) {
            x[k] = 1.0f / x[k];
            __builtin_amdgcn_sched_barrier(0);  // one at a time: this path must not set the register count
        }
    }
}

// Equations that quots_rn puts behind one branch.  All 16 at once: 139
// registers in place of 129 (split_kernels.hpp, stage 3 of 16 x 16), and 256
// in place of 233 on 32 equations per lane.
constexpr int kQuotChunk = 8;

// n / x for y = recip_short(x), rounded as IEEE division does, where n is zero
// or |n| and |x| lie in [2^-60, 2^60].  y is then 1 / x rounded to nearest,
// and one correction of n y rounds the quotient right: so for every pair of
// significands (all 2^46 compared with n / x; the powers of two only scale,
// nothing here being subnormal or infinite).  The fixup keeps the sign of a
// zero and the results of infinities and NaNs.
__device__ __forceinline__ float quot_short(float n, float x, float y) {
    const float q = n * y;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-x, q, n), y, q), x, n);
}

// a[k], c[k], d[k] -> their quotients by b[k], rounded as IEEE division does
// (src/ptpr.hpp:80-90): three quotients of one reciprocal, 25 issue slots per
// equation against 42 for three divisions, range tests included.  Eight
// equations at a time share one branch for the wavefront.
template <int E>
__device__ __forceinline__ void quots_rn(const float (&a)[E], const float (&c)[E], const float (&d)[E],
                                         const float (&b)[E], float (&A)[E], float (&C)[E], float (&R)[E]) {
    constexpr int W = E < kQuotChunk ? E : kQuotChunk;
    // 2 |v| as a bit pattern, a zero above all others
    auto key = [](float v) { return (__builtin_bit_cast(unsigned, v) << 1) - 1u; };
    auto least = [](unsigned u, unsigned v) { return u < v ? u : v; };
#pragma unroll
    for (int k0 = 0; k0 < E; k0 += W) {
        float mx = 0.0f, bn = __builtin_fabsf(b[k0]);
        unsigned kn = 0xffffffffu;
#pragma unroll
        for (int k = k0; k < k0 + W; k++) {
            mx = __builtin_fmaxf(__builtin_fmaxf(mx, __builtin_fabsf(a[k])), __builtin_fabsf(c[k]));
            mx = __builtin_fmaxf(__builtin_fmaxf(mx, __builtin_fabsf(d[k])), __builtin_fabsf(b[k]));
            bn = __builtin_fminf(bn, __builtin_fabsf(b[k]));
            kn = least(kn, least(key(a[k]), least(key(c[k]), key(d[k]))));
        }
        const bool plain = mx <= 0x1p60f && bn >= 0x1p-60f && kn >= key(0x1p-60f);
        if (__ballot(!plain) == 0) {
#pragma unroll
            for (int k = k0; k < k0 + W; k++) {
                const float y = recip_short(b[k]);
                A[k] = quot_short(a[k], b[k], y);
                C[k] = quot_short(c[k], b[k], y);
                R[k] = quot_short(d[k], b[k], y);
            }
        } else {
#pragma unroll
            for (int k = k0; k < k0 + W; k++) {
                A[k] = a[k] / b[k];
                C[k] = c[k] / b[k];
                R[k] = d[k] / b[k];
                __builtin_amdgcn_sched_barrier(0);  // one at a time: this path must not set the register count
            }
        }
    }
}

// The two halves of an exact pcr_update (tpr_device.hpp), so that several
// rows' reciprocals share one range test and branch in between: the
// denominator and the right-hand side's sum, and the row from the inverse.
__device__ __forceinline__ void pcr_sums(Eq k, Eq kl, Eq kr, bool hasL, bool hasR, float& den, float& rn) {
    const float t1 = hasL ? (1.0f - kl.c * k.a) : 1.0f;
    den = hasR ? (t1 - kr.a * k.c) : t1;
    rn = hasL ? (k.r - kl.r * k.a) : k.r;
    rn = settled(hasR ? (rn - kr.r * k.c) : rn);
}
__device__ __forceinline__ Eq pcr_row(Eq k, Eq kl, Eq kr, bool hasL, bool hasR, float inv, float rn) {
    return Eq{hasL ? (-inv * kl.a) * k.a : inv * k.a, hasR ? (-inv * kr.c) * k.c : inv * k.c, inv * rn};
}

// One level on the blocked layout, u = U < E.
template <int E, int L, int U>
__device__ __forceinline__ void exact_level_blocked(float (&Ap)[E], float (&Cp)[E], float (&R)[E], int l) {
    float inv[E], rn[E];
#pragma unroll
    for (int j = 0; j < E; j++) {
        const bool lx = j < U, rx = j + U >= E;  // partner in the lane before / after
        const float ka = Ap[j], kc = Cp[j];
        const int jl = lx ? E - U + j : j - U, jr = rx ? j + U - E : j + U;
        float p1, p2, p3, p4;
        if (lx) {
            exact_mul_up<L, 1>(Cp[jl], R[jl], ka, l, p1, p3);
        } else {
            p1 = Cp[jl] * ka;
            p3 = R[jl] * ka;
        }
        if (rx) {
            exact_mul_dn<L, 1>(Ap[jr], R[jr], kc, l, p2, p4);
        } else {
            p2 = Ap[jr] * kc;
            p4 = R[jr] * kc;
        }
        inv[j] = (1.0f - p1) - p2;
        rn[j] = settled((R[j] + p3) + p4);
    }
    recips_rn<E>(inv);
    // in place: the partners in other lanes first, then each array in the
    // order that reads a register before it is overwritten
    float ul[U], vr[U];
#pragma unroll
    for (int j = 0; j < U; j++) {
        ul[j] = exact_keep_up<L, 1>(Ap[E - U + j], inv[j], l);
        vr[j] = exact_keep_dn<L, 1>(Cp[j], inv[E - U + j], l);
    }
#pragma unroll
    for (int j = E - 1; j >= 0; j--) Ap[j] = (j < U ? ul[j < U ? j : 0] : inv[j] * Ap[j < U ? 0 : j - U]) * Ap[j];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < E; j++)
        Cp[j] = (j + U >= E ? vr[j + U >= E ? j + U - E : 0] : inv[j] * Cp[j + U >= E ? 0 : j + U]) * Cp[j];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < E; j++) R[j] = inv[j] * rn[j];
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (2 * U < E) exact_level_blocked<E, L, 2 * U>(Ap, Cp, R, l);
}

// One level between the two layouts' reach: the partner of every register is
// the same register D lanes away.
template <int E, int L, int D>
__device__ __forceinline__ void exact_level_lanes(float (&Ap)[E], float (&Cp)[E], float (&R)[E], int l) {
    float inv[E], rn[E];
#pragma unroll
    for (int j = 0; j < E; j++) {
        const float ka = Ap[j], kc = Cp[j];
        float p1, p2, p3, p4;
        exact_mul_up<L, D>(Cp[j], R[j], ka, l, p1, p3);
        exact_mul_dn<L, D>(Ap[j], R[j], kc, l, p2, p4);
        inv[j] = (1.0f - p1) - p2;
        rn[j] = settled((R[j] + p3) + p4);
    }
    recips_rn<E>(inv);
#pragma unroll
    for (int j = 0; j < E; j++) {
        Ap[j] = exact_keep_up<L, D>(Ap[j], inv[j], l) * Ap[j];
        Cp[j] = exact_keep_dn<L, D>(Cp[j], inv[j], l) * Cp[j];
        R[j] = inv[j] * rn[j];
    }
    if constexpr (2 * D * E < L) exact_level_lanes<E, L, 2 * D>(Ap, Cp, R, l);
}

// One level on the strided layout: partners K registers away.
template <int E, int K>
__device__ __forceinline__ void exact_level_strided(float (&Ap)[E], float (&Cp)[E], float (&R)[E]) {
    float inv[E], rn[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const bool hl = e >= K, hr = e + K < E;
        float den = 1.0f, r = R[e];
        if (hl) {
            den = den - Cp[hl ? e - K : 0] * Ap[e];
            r = r + R[hl ? e - K : 0] * Ap[e];
        }
        if (hr) {
            den = den - Ap[hr ? e + K : 0] * Cp[e];
            r = r + R[hr ? e + K : 0] * Cp[e];
        }
        inv[e] = den;
        rn[e] = settled(r);
    }
    recips_rn<E>(inv);
#pragma unroll
    for (int e = E - 1; e >= 0; e--) Ap[e] = (e >= K ? inv[e] * Ap[e >= K ? e - K : 0] : inv[e]) * Ap[e];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < E; e++) Cp[e] = (e + K < E ? inv[e] * Cp[e + K < E ? e + K : 0] : inv[e]) * Cp[e];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < E; e++) R[e] = inv[e] * rn[e];
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (2 * K < E) exact_level_strided<E, 2 * K>(Ap, Cp, R);
}

// Shapes that run this way (E = 4 and below, and TPR, keep the register form).
template <int E, int L>
constexpr bool kExactTurn = (E == 8 || E == 16 || E == 32) && (L == 16 || L == 32 || L == 64) && L >= E;

// Stage 1 from the normalised equations, blocked; leaves A, C, R strided.
// The slice's first row is in register 0 of its first lane and its last in
// register E - 1 of its last lane, in both layouts.  area: the wavefront's 68
// E floats of LDS.  Every lane of the wavefront calls this.
template <int E, int L>
__device__ __forceinline__ void exact_stage1_turned(float (&A)[E], float (&C)[E], float (&R)[E], int l, float* area,
                                                    int lane) {
#pragma unroll
    for (int e = 0; e < E; e++) {
        A[e] = -A[e];
        C[e] = -C[e];
    }
    exact_level_blocked<E, L, 1>(A, C, R, l);
    if constexpr (E < L) exact_level_lanes<E, L, 1>(A, C, R, l);
    turn_strided<E, L>(A, area, lane);
    turn_strided<E, L>(C, area, lane);
    turn_strided<E, L>(R, area, lane);
    exact_level_strided<E, 1>(A, C, R);
#pragma unroll
    for (int e = 0; e < E; e++) {
        A[e] = -A[e];
        C[e] = -C[e];
    }
}

}  // namespace tprh
