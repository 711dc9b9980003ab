// serve.hip -- the serving loop's batch kernel: systems of different sizes,
// several right-hand sides per matrix, in one launch.
//
// Same scheduling as the uneven-batch kernels (work items of one size class;
// workgroups of 256 lanes, or persistent ones of 1024); each system entry
// names its own matrix, right-hand side and answer in the server's arena, so
// every right-hand side of a request reads the request's one resident copy
// of a, b, c (HBM traffic 12 B per matrix equation + 8 B per right-hand-side
// equation when the coefficients stay in cache between its systems).
#include <hip/hip_runtime.h>

#include <atomic>

#include "launch_serve.hpp"
#include "solve_slot.hpp"

namespace tprh {

template <int METHOD, int MODE, int BLOCK>
__device__ __forceinline__ void run_serve_item(const UnevenTask& tk, const ServeSys* __restrict__ sys,
                                               float* __restrict__ base, float* lds) {
    const int slot = threadIdx.x >> tk.lg_lanes;
    const int t = threadIdx.x & ((1 << tk.lg_lanes) - 1);
    const ServeSys e = sys[tk.first + (slot < tk.count ? slot : 0)];
    switch (tk.shape) {
#define TPRH_SERVE_CASE(ID, EE, LL)                                                                              \
    case ID: {                                                                                                   \
        const size_t n = (size_t)tk.m * (EE * LL);                                                               \
        const size_t off = (size_t)t * EE;                                                                       \
        const SlotAt at{(size_t)e.coef + off, (size_t)e.rhs + off, (size_t)e.x + off};                           \
        solve_slot<METHOD, MODE, true, EE, LL, BLOCK>(tk.m, tk.lg_lanes, tk.count, base, base + n, base + 2 * n, \
                                                      base, base, at, lds);                                      \
        break;                                                                                                   \
    }
        TPRH_UNEVEN_SHAPES(TPRH_SERVE_CASE)
#undef TPRH_SERVE_CASE
        default:
            break;
    }
}

// counter NULL: a workgroup per item.
template <int METHOD, int MODE>
__global__ __launch_bounds__(kSlotBig) void serve_kernel(const UnevenTask* __restrict__ tasks, int ntasks,
                                                         int* __restrict__ counter, const ServeSys* __restrict__ sys,
                                                         float* __restrict__ base) {
    extern __shared__ float lds[];
    __shared__ int item;
    if (threadIdx.x == 0) item = counter ? atomicAdd(counter, 1) : (int)blockIdx.x;
    __syncthreads();
    int it = __builtin_amdgcn_readfirstlane(item);
    while (it < ntasks) {  // uniform: every workgroup leaves once the items are gone
        // the next ticket is asked for now and read after this item, so the
        // device-coherent counter's latency hides under the item's loads
        int nxt = ntasks;
        if (threadIdx.x == 0 && counter) nxt = next_ticket(counter);
        run_serve_item<METHOD, MODE, kSlotBig>(tasks[it], sys, base, lds);
        __syncthreads();  // the item's LDS rows are read before the next item writes them;
                          // every thread has read `item` before it is rewritten
        if (threadIdx.x == 0) item = nxt;
        __syncthreads();
        it = __builtin_amdgcn_readfirstlane(item);
    }
}

// One item per workgroup.
template <int METHOD, int MODE>
__global__ __launch_bounds__(kSlotTile, 4) void serve_tile_kernel(const UnevenTask* __restrict__ tasks,
                                                                  const ServeSys* __restrict__ sys,
                                                                  float* __restrict__ base) {
    extern __shared__ float lds[];
    run_serve_item<METHOD, MODE, kSlotTile>(tasks[blockIdx.x], sys, base, lds);
}

namespace {

template <int METHOD, int MODE>
hipError_t allow_big_lds() {
    static std::atomic<unsigned long long> set{0};
    if (slot_big_lds(METHOD, MODE) <= 65536) return hipSuccess;
    return ensure_lds_limit(reinterpret_cast<const void*>(serve_kernel<METHOD, MODE>), (int)slot_big_lds(METHOD, MODE),
                            set);
}

template <int METHOD, int MODE>
hipError_t launch_serve_t(const ServeLaunch& p, hipStream_t stream) {
    if (p.block == kSlotBig) {
        hipError_t e = allow_big_lds<METHOD, MODE>();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((serve_kernel<METHOD, MODE>), dim3(p.grid), dim3(kSlotBig), slot_big_lds(METHOD, MODE),
                           stream, p.tasks, p.ntasks, p.ntasks > p.grid ? p.counter : nullptr, p.sys, p.base);
    } else {
        hipLaunchKernelGGL((serve_tile_kernel<METHOD, MODE>), dim3(p.ntasks), dim3(kSlotTile),
                           slot_lds_bytes(kSlotTile, true), stream, p.tasks, p.sys, p.base);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_serve(int method, int mode, const ServeLaunch& p, hipStream_t stream) {
    if (method == 0) return mode == kExact ? launch_serve_t<0, kExact>(p, stream) : launch_serve_t<0, kFast>(p, stream);
    return mode == kExact ? launch_serve_t<1, kExact>(p, stream) : launch_serve_t<1, kFast>(p, stream);
}

hipError_t serve_occupancy(int method, int mode, size_t lds_bytes, int* blocks_per_cu) {
    const void* f;
    if (method == 0) f = mode == kExact ? reinterpret_cast<const void*>(serve_kernel<0, kExact>)
                                        : reinterpret_cast<const void*>(serve_kernel<0, kFast>);
    else f = mode == kExact ? reinterpret_cast<const void*>(serve_kernel<1, kExact>)
                            : reinterpret_cast<const void*>(serve_kernel<1, kFast>);
    if (method == 0 && mode == kExact) {
        hipError_t e = allow_big_lds<0, kExact>();
        if (e != hipSuccess) return e;
    }
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, f, kSlotBig, lds_bytes);
}

}  // namespace tprh
