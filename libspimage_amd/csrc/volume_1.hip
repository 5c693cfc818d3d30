// Instances of the two-pass volume kernels (volume.h).
#include "volume.h"

namespace spx {
const VolOps* vol_ops_1(int L) {
  static const VolOps v80 = vol_ops_of<80>();
  static const VolOps v96 = vol_ops_of<96>();
  static const VolOps v240 = vol_ops_of<240>();
  switch (L) {
    case 80: return &v80;
    case 96: return &v96;
    case 240: return &v240;
  }
  return nullptr;
}
}  // namespace spx
