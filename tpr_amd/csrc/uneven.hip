// uneven.hip -- batches of systems of different sizes in one launch.
//
// A plan (built on the host, see capi.hip) sorts the systems into size
// classes, gives every class a slice size s and slice shape (E, L) from a
// per-class table (the autotuner's), and cuts each class into work items of
// as many systems as one workgroup holds: 256 lanes where all of the plan's
// systems fit them, one workgroup per item, else 1024 lanes in a persistent
// kernel.  That one keeps one workgroup per resident slot.  Up to kSweepRounds
// items each it takes them in turn; beyond, each workgroup takes the next from
// an atomic counter (items are ordered largest systems first) and asks for its
// next ticket as it starts an item, so the counter's latency hides under the
// item.  Every system's result
// depends only on its own size class's (s, E, L), never on the batch around
// it.
#include <hip/hip_runtime.h>

#include <atomic>

#include "launch_uneven.hpp"
#include "slice_solvers.hpp"
#include "solve_slot.hpp"

namespace tprh {

template <int METHOD, int MODE, bool HAS_B, int E, int L, int BLOCK>
__device__ __forceinline__ void run_task(const UnevenTask& tk, const int* __restrict__ sys_list,
                                         const long long* __restrict__ offsets, const float* __restrict__ a,
                                         const float* __restrict__ b, const float* __restrict__ c,
                                         const float* __restrict__ d, float* __restrict__ x, float* lds) {
    const int slot = threadIdx.x >> tk.lg_lanes;
    const int sys = sys_list[tk.first + (slot < tk.count ? slot : 0)];
    const size_t at = (size_t)offsets[sys] + (size_t)(threadIdx.x & ((1 << tk.lg_lanes) - 1)) * E;
    solve_slot<METHOD, MODE, HAS_B, E, L, BLOCK>(tk.m, tk.lg_lanes, tk.count, a, b, c, d, x, SlotAt{at, at, at}, lds);
}

template <int METHOD, int MODE, bool HAS_B, int BLOCK>
__device__ __forceinline__ void run_shape(const UnevenTask& tk, const int* __restrict__ sys_list,
                                          const long long* __restrict__ offsets, const float* __restrict__ a,
                                          const float* __restrict__ b, const float* __restrict__ c,
                                          const float* __restrict__ d, float* __restrict__ x, float* lds) {
    switch (tk.shape) {
#define TPRH_UNEVEN_CASE(ID, EE, LL)                                                              \
    case ID:                                                                                      \
        run_task<METHOD, MODE, HAS_B, EE, LL, BLOCK>(tk, sys_list, offsets, a, b, c, d, x, lds); \
        break;
        TPRH_UNEVEN_SHAPES(TPRH_UNEVEN_CASE)
#undef TPRH_UNEVEN_CASE
        default:
            break;
    }
}

__global__ void zero_counter_kernel(int* counter) { *counter = 0; }

// counter NULL: workgroup k takes the items k, k + grid, ...
template <int METHOD, int MODE, bool HAS_B>
__global__ __launch_bounds__(kSlotBig) void uneven_kernel(const UnevenTask* __restrict__ tasks, int ntasks,
                                                          int* __restrict__ counter, const int* __restrict__ sys_list,
                                                          const long long* __restrict__ offsets,
                                                          const float* __restrict__ a, const float* __restrict__ b,
                                                          const float* __restrict__ c, const float* __restrict__ d,
                                                          float* __restrict__ x) {
    extern __shared__ float lds[];
    __shared__ int item;
    if (threadIdx.x == 0) item = counter ? atomicAdd(counter, 1) : (int)blockIdx.x;
    __syncthreads();
    int it = __builtin_amdgcn_readfirstlane(item);
    while (it < ntasks) {  // uniform: every workgroup leaves once the items are gone
        // the next item's ticket is asked for now and read after this item:
        // the counter is device-coherent, its answer takes microseconds
        // behind the memory traffic, and this item's loads now cover that
        // wait (a workgroup holds at most two tickets; items are independent)
        int nxt = it + (int)gridDim.x;
        if (threadIdx.x == 0 && counter) nxt = next_ticket(counter);
        run_shape<METHOD, MODE, HAS_B, kSlotBig>(tasks[it], sys_list, offsets, a, b, c, d, x, lds);
        __syncthreads();  // the item's LDS rows are read before the next item writes them;
                          // every thread has read `item` before it is rewritten
        if (threadIdx.x == 0) item = nxt;
        __syncthreads();
        it = __builtin_amdgcn_readfirstlane(item);
    }
}

// One item per workgroup.
template <int METHOD, int MODE, bool HAS_B>
__global__ __launch_bounds__(kSlotTile, 4) void uneven_tile_kernel(const UnevenTask* __restrict__ tasks,
                                                                   const int* __restrict__ sys_list,
                                                                   const long long* __restrict__ offsets,
                                                                   const float* __restrict__ a,
                                                                   const float* __restrict__ b,
                                                                   const float* __restrict__ c,
                                                                   const float* __restrict__ d,
                                                                   float* __restrict__ x) {
    extern __shared__ float lds[];
    run_shape<METHOD, MODE, HAS_B, kSlotTile>(tasks[blockIdx.x], sys_list, offsets, a, b, c, d, x, lds);
}

namespace {

// Items per workgroup up to which they are taken in turn: the counter's clear
// is a launch of 5 us, and what the counter balances grows with the items.
// Systems of 256 .. 16384, counter -> in turn: 1300 (1.5 items) 38.9 -> 34.1
// us, 2500 (2.8) 67.2 -> 66.1, 4000 (4.4) 94.4 -> 103, 20000 (22) 385 -> 404.
constexpr int kSweepRounds = 3;

template <int METHOD, int MODE, bool HAS_B>
hipError_t allow_big_lds() {
    static std::atomic<unsigned long long> set{0};
    if (slot_big_lds(METHOD, MODE) <= 65536) return hipSuccess;
    return ensure_lds_limit(reinterpret_cast<const void*>(uneven_kernel<METHOD, MODE, HAS_B>),
                            (int)slot_big_lds(METHOD, MODE), set);
}

template <int METHOD, int MODE, bool HAS_B>
hipError_t launch_uneven_t(const UnevenLaunch& p, hipStream_t stream) {
    if (p.block == kSlotBig) {
        hipError_t e = allow_big_lds<METHOD, MODE, HAS_B>();
        if (e != hipSuccess) return e;
        int* counter = p.ntasks > kSweepRounds * (long long)p.grid ? p.counter : nullptr;
        if (counter) hipLaunchKernelGGL(zero_counter_kernel, dim3(1), dim3(1), 0, stream, counter);
        hipLaunchKernelGGL((uneven_kernel<METHOD, MODE, HAS_B>), dim3(p.grid), dim3(kSlotBig),
                           slot_big_lds(METHOD, MODE), stream, p.tasks, p.ntasks, counter, p.sys_list, p.offsets, p.a,
                           p.b, p.c, p.d, p.x);
    } else {
        hipLaunchKernelGGL((uneven_tile_kernel<METHOD, MODE, HAS_B>), dim3(p.ntasks), dim3(kSlotTile),
                           slot_lds_bytes(kSlotTile, true), stream, p.tasks, p.sys_list, p.offsets, p.a, p.b, p.c,
                           p.d, p.x);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_uneven(int method, int mode, const UnevenLaunch& p, hipStream_t stream) {
    const bool hb = p.b != nullptr;
    if (method == 0) {
        if (mode == kExact) return hb ? launch_uneven_t<0, kExact, true>(p, stream) : launch_uneven_t<0, kExact, false>(p, stream);
        return hb ? launch_uneven_t<0, kFast, true>(p, stream) : launch_uneven_t<0, kFast, false>(p, stream);
    }
    if (mode == kExact) return hb ? launch_uneven_t<1, kExact, true>(p, stream) : launch_uneven_t<1, kExact, false>(p, stream);
    return hb ? launch_uneven_t<1, kFast, true>(p, stream) : launch_uneven_t<1, kFast, false>(p, stream);
}

hipError_t uneven_occupancy(int method, int mode, int* blocks_per_cu) {
    const void* f;
    if (method == 0) f = mode == kExact ? reinterpret_cast<const void*>(uneven_kernel<0, kExact, true>)
                                        : reinterpret_cast<const void*>(uneven_kernel<0, kFast, true>);
    else f = mode == kExact ? reinterpret_cast<const void*>(uneven_kernel<1, kExact, true>)
                            : reinterpret_cast<const void*>(uneven_kernel<1, kFast, true>);
    if (method == 0 && mode == kExact) {
        hipError_t e = allow_big_lds<0, kExact, true>();
        if (e != hipSuccess) return e;
    }
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, f, kSlotBig, slot_big_lds(method, mode));
}

}  // namespace tprh
