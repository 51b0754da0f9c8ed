// The four-wide traversal kernels for Wald triangles.
#include "wide_trace.h"

namespace mh {

int launch_wide_table_wald(const DevScene& sc, const BatchLaunch& bl, hipStream_t s) {
  return launch_wide_table<1>(sc, bl, s);
}

int launch_wide_one_wald(const DevScene& sc, const BatchDev& rays, const LaunchCfg& cfg,
                       hipStream_t s) {
  return launch_wide_one<1>(sc, rays, cfg, s);
}

}  // namespace mh
