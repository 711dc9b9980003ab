// exact_div.hip -- a diagnostic build (libtpr_diag.so, not part of the
// solver library): checks the solver's short reciprocal (recip_rn in
// tpr_amd/csrc/tpr_device.hpp) against IEEE division, 1.0f / x, for every
// one of the 2^32 float bit patterns x on the GPU.  Equal means the same
// bits, or both NaN.  Counts go to counts[0] (recip_rn, the guarded form the
// kernels use), counts[1] (the unguarded four-instruction sequence) and,
// for the unguarded one, counts[2] (x subnormal), counts[3]
// (2^-126 <= |x| < 2^-125 or |x| > 2^126) and counts[4] (the rest); up to 64
// patterns where the guarded form differs go to bad[].
#include <hip/hip_runtime.h>

#include "../csrc/exact_rows.hpp"
#include "../csrc/tpr_device.hpp"

namespace {

__device__ bool same(float a, float b) {
    return __builtin_bit_cast(unsigned, a) == __builtin_bit_cast(unsigned, b) || (a != a && b != b);
}

__global__ void recip_check_kernel(unsigned long long* __restrict__ counts, unsigned* __restrict__ bad) {
    const unsigned long long total = 1ull << 32;
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    unsigned long long c0 = 0, c1 = 0, c2 = 0, c3 = 0, c4 = 0;
    for (unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const unsigned u = (unsigned)i;
        const float x = __builtin_bit_cast(float, u);
        const float ref = 1.0f / x;
        if (!same(tprh::recip_rn(x), ref)) {
            c0++;
            const unsigned long long k = atomicAdd(&counts[5], 1ull);
            if (k < 64) bad[k] = u;
        }
        if (!same(tprh::recip_rn_unguarded(x), ref)) {
            c1++;
            const unsigned ax = u & 0x7fffffffu;
            if (ax < 0x00800000u) c2++;
            else if (ax < 0x01000000u || ax > 0x7e800000u) c3++;
            else c4++;
        }
    }
    if (c0) atomicAdd(&counts[0], c0);
    if (c1) atomicAdd(&counts[1], c1);
    if (c2) atomicAdd(&counts[2], c2);
    if (c3) atomicAdd(&counts[3], c3);
    if (c4) atomicAdd(&counts[4], c4);
}

// recip_short (tpr_amd/csrc/exact_rows.hpp) against 1.0f / x for every float
// with 2^-126 <= |x| <= 2^126 and every NaN: the inputs for which recips_rn
// takes it.  counts[0]: differences; counts[1]: inputs compared.
__global__ void recip_short_check_kernel(unsigned long long* __restrict__ counts) {
    const unsigned long long total = 1ull << 32;
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    unsigned long long differ = 0, seen = 0;
    for (unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const float x = __builtin_bit_cast(float, (unsigned)i);
        const float ax = __builtin_fabsf(x);
        if (x == x && !(ax >= 0x1p-126f && ax <= 0x1p126f)) continue;
        seen++;
        if (!same(tprh::recip_short(x), 1.0f / x)) differ++;
    }
    if (differ) atomicAdd(&counts[0], differ);
    atomicAdd(&counts[1], seen);
}

// quot_short against n / x: `blocks` workgroups, workgroup k with the
// significand first + k * stride of x, all 2^23 of n, at random powers of two
// that keep both inside [2^-60, 2^60], and both signs.  counts[0]:
// differences; counts[1]: pairs compared.
__global__ void quot_short_check_kernel(unsigned first, unsigned stride, unsigned long long* __restrict__ counts) {
    const unsigned sx = (first + blockIdx.x * stride) & 0x7fffffu;
    unsigned long long differ = 0, seen = 0;
    unsigned rnd = sx * 2654435761u + threadIdx.x * 40503u + 12345u;
    for (unsigned sn = threadIdx.x; sn < (1u << 23); sn += blockDim.x) {
        rnd = rnd * 1664525u + 1013904223u;
        const unsigned ex = 67 + (rnd >> 8) % 120, en = 67 + (rnd >> 16) % 120;  // 2^-60 .. 2^59
        const float x = __builtin_bit_cast(float, (rnd & 0x80000000u) | ex << 23 | sx);
        const float n = __builtin_bit_cast(float, (rnd << 1 & 0x80000000u) | en << 23 | sn);
        seen++;
        if (!same(tprh::quot_short(n, x, tprh::recip_short(x)), n / x)) differ++;
    }
    if (differ) atomicAdd(&counts[0], differ);
    atomicAdd(&counts[1], seen);
}

// quots_rn against the division of its operands, one lane's eight equations:
// ops holds 4 x 8 x 64 floats per workgroup (a, c, d, b of 64 lanes by 8).
__global__ void quots_check_kernel(const float* __restrict__ ops, unsigned long long* __restrict__ counts) {
    const float* p = ops + (size_t)blockIdx.x * 4 * 8 * 64 + threadIdx.x * 8;
    float v[4][8], A[8], C[8], R[8];
    for (int w = 0; w < 4; w++)
        for (int k = 0; k < 8; k++) v[w][k] = p[w * 8 * 64 + k];
    tprh::quots_rn<8>(v[0], v[1], v[2], v[3], A, C, R);
    unsigned long long differ = 0;
    for (int k = 0; k < 8; k++) {
        differ += !same(A[k], v[0][k] / v[3][k]);
        differ += !same(C[k], v[1][k] / v[3][k]);
        differ += !same(R[k], v[2][k] / v[3][k]);
    }
    if (differ) atomicAdd(&counts[0], differ);
    atomicAdd(&counts[1], 24ull);
}

}  // namespace

// Both return a hipError_t; counts: 2 zeroed words.
extern "C" int tprh_diag_quot_short_check(int blocks, unsigned first, unsigned stride, unsigned long long* counts,
                                          void* stream) {
    hipLaunchKernelGGL(quot_short_check_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, first, stride, counts);
    return (int)hipGetLastError();
}
extern "C" int tprh_diag_quots_check(const float* ops, int blocks, unsigned long long* counts, void* stream) {
    hipLaunchKernelGGL(quots_check_kernel, dim3(blocks), dim3(64), 0, (hipStream_t)stream, ops, counts);
    return (int)hipGetLastError();
}

// counts: 2 zeroed words.  Returns a hipError_t.
extern "C" int tprh_diag_recip_short_check(unsigned long long* counts, void* stream) {
    hipLaunchKernelGGL(recip_short_check_kernel, dim3(8192), dim3(256), 0, (hipStream_t)stream, counts);
    return (int)hipGetLastError();
}

// counts: 6 zeroed words (the last one counts recorded patterns); bad: 64
// words.  Returns a hipError_t.
extern "C" int tprh_diag_recip_check(unsigned long long* counts, unsigned* bad, void* stream) {
    hipLaunchKernelGGL(recip_check_kernel, dim3(8192), dim3(256), 0, (hipStream_t)stream, counts, bad);
    return (int)hipGetLastError();
}
