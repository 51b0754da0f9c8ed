// The four-wide traversal kernels for Kensler-Shirley triangles.
#include "wide_trace.h"

namespace mh {

int launch_wide_table_ks(const DevScene& sc, const BatchLaunch& bl, hipStream_t s) {
  return launch_wide_table<0>(sc, bl, s);
}

int launch_wide_one_ks(const DevScene& sc, const BatchDev& rays, const LaunchCfg& cfg,
                       hipStream_t s) {
  return launch_wide_one<0>(sc, rays, cfg, s);
}

}  // namespace mh
