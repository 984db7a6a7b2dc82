// Builds of the runtime-length pass for double (hmi_generic.h).
#include "hmi_generic.h"

namespace hmi {

hipError_t launch_mixed_f64(const pass_args &a, const mixed_plan &g, int threads, long long nblocks, size_t lds_bytes,
                           hipStream_t s) {
    return generic_builds<double>::launch(a, g, threads, nblocks, lds_bytes, s);
}

}  // namespace hmi
