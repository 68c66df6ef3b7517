// The lanes per face that a multi-mesh run's depth passes use and those of the autotuner's trials of its
// meshes (gvv_kernels.hpp), over item counts on both sides of every limit: a line "items lanes
// batched_lanes" each.  Host only.
#include <hip/hip_runtime.h>
#include <cstdio>
#include "../gvv-differentiable-cuda-renderer_amd/csrc/gvv_kernels.hpp"
int main() {
  for (long long n : {1ll, 65536ll, 65537ll, 262144ll, 262145ll, 2097152ll, 2097153ll, 1ll << 40})
    printf("%lld %d %d %d\n", n, gvv::raster_lanes(gvv::shared_raster_items(n, false)),
           gvv::raster_lanes(gvv::shared_raster_items(n, true)), gvv::kBatchedLanes);
  return 0;
}
