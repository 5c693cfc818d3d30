// Instances of the two-pass volume kernels (volume.h).
#include "volume.h"

namespace spx {
const VolOps* vol_ops_3(int L) {
  static const VolOps v144 = vol_ops_of<144>();
  static const VolOps v160 = vol_ops_of<160>();
  switch (L) {
    case 144: return &v144;
    case 160: return &v160;
  }
  return nullptr;
}
}  // namespace spx
