// Builds of the fused two-axis pass for double (hmi_plane.h).
#include "hmi_plane.h"

namespace hmi {

hipError_t launch_plane_f64(const plane_args &a, int threads, long long nblocks, size_t lds_bytes, hipStream_t s) {
    return plane_builds<double>::launch(a, threads, nblocks, lds_bytes, s);
}

hipError_t launch_batch_fused_f64(bool xy, const batch_args &b, int threads, int nblocks, size_t lds_bytes, hipStream_t s) {
    return launch_batch_builds<double>(xy, b, threads, nblocks, lds_bytes, s);
}

}  // namespace hmi
