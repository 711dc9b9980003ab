// batched_ptpr.hip -- the PTPR instantiations of the batched kernel.
#include "batched_impl.hpp"

namespace tprh {

hipError_t launch_batched_ptpr(int mode, const BatchArgs& p, int E, int L, hipStream_t stream) {
    if (mode == kFast && fast_rows_16(E, L, p.n)) {
        // slices of several DPP rows (fast_rows_16, launch.hpp): the two-level
        // stage 1 on rows of 16 lanes x 16 equations, every row of the system
        // one row of its reduced system
        BatchArgs q = p;
        q.m = p.n / 256;
        return launch_batched_method<0>(mode, q, 16, 16, stream);
    }
    return launch_batched_method<0>(mode, p, E, L, stream);
}

hipError_t launch_batched(int method, int mode, const BatchArgs& p, int E, int L, hipStream_t stream) {
    return method == 0 ? launch_batched_ptpr(mode, p, E, L, stream) : launch_batched_tpr(mode, p, E, L, stream);
}

}  // namespace tprh
