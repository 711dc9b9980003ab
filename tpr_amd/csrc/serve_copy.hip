// serve_copy.hip -- the serving loop's copies of callers' right-hand sides
// into the arena, one launch for all of a batch's.
//
// One hipMemcpyAsync per request costs the worker a few microseconds of host
// time and the batch's stream 2 to 4.5 us of device time, whatever its size
// (a request's right-hand sides are 2 KB to 8 MB): 48 requests took 96
// copies, in and out, 0.3 of the burst's 0.44 ms.  Here one kernel copies
// every run that lies in this device's memory, 4096 floats per workgroup, at
// the rate of a device copy; answers for buffers in this device's memory are
// written there by the solve itself (server.hip).  48 requests in a burst: 0.44
// -> 0.21 ms.
#include <hip/hip_runtime.h>

#include "launch_serve.hpp"

namespace tprh {

__global__ __launch_bounds__(256) void copy_runs_kernel(const CopyRun* __restrict__ runs, int nruns) {
    // the run of this workgroup's chunk: the last one that starts at or before it
    const int b = blockIdx.x;
    int lo = 0, hi = nruns - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (runs[mid].first <= b) lo = mid;
        else hi = mid - 1;
    }
    const CopyRun r = runs[lo];
    const long long at = (long long)(b - r.first) * kCopyChunk;
    const float* src = r.src + at;
    float* dst = r.dst + at;
    const int left = (int)(r.count - at < kCopyChunk ? r.count - at : kCopyChunk);
    // whole 16-byte pieces where both sides are aligned; callers' buffers
    // need not be
    if ((((size_t)src | (size_t)dst) & 15) == 0) {
        const int pieces = left >> 2;
        for (int i = threadIdx.x; i < pieces; i += 256)
            reinterpret_cast<float4*>(dst)[i] = reinterpret_cast<const float4*>(src)[i];
        for (int i = (pieces << 2) + threadIdx.x; i < left; i += 256) dst[i] = src[i];
    } else {
        for (int i = threadIdx.x; i < left; i += 256) dst[i] = src[i];
    }
}

hipError_t launch_copy_runs(const CopyRun* runs, int nruns, int chunks, hipStream_t stream) {
    hipLaunchKernelGGL(copy_runs_kernel, dim3(chunks), dim3(256), 0, stream, runs, nruns);
    return hipGetLastError();
}

bool device_allocation(const void* p, int device, size_t* lo, size_t* hi) {
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();  // not memory the runtime knows
        return false;
    }
    if (at.type != hipMemoryTypeDevice || at.device != device || at.isManaged) return false;
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, const_cast<void*>(p)) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    *lo = reinterpret_cast<size_t>(base);
    *hi = *lo + size;
    return true;
}

}  // namespace tprh
