// Builds of the fused two-axis pass for float (hmi_plane.h).
#include "hmi_plane.h"

namespace hmi {

hipError_t launch_plane_f32(const plane_args &a, int threads, long long nblocks, size_t lds_bytes, hipStream_t s) {
    return plane_builds<float>::launch(a, threads, nblocks, lds_bytes, s);
}

hipError_t launch_batch_fused_f32(bool xy, const batch_args &b, int threads, int nblocks, size_t lds_bytes, hipStream_t s) {
    return launch_batch_builds<float>(xy, b, threads, nblocks, lds_bytes, s);
}

}  // namespace hmi
