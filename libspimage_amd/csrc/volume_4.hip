// Instances of the two-pass volume kernels (volume.h).
#include "volume.h"

namespace spx {
const VolOps* vol_ops_4(int L) {
  static const VolOps v192 = vol_ops_of<192>();
  static const VolOps v200 = vol_ops_of<200>();
  switch (L) {
    case 192: return &v192;
    case 200: return &v200;
  }
  return nullptr;
}
}  // namespace spx
