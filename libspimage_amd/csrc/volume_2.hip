// Instances of the two-pass volume kernels (volume.h).
#include "volume.h"

namespace spx {
const VolOps* vol_ops_2(int L) {
  static const VolOps v120 = vol_ops_of<120>();
  static const VolOps v128 = vol_ops_of<128>();
  static const VolOps v216 = vol_ops_of<216>();
  switch (L) {
    case 120: return &v120;
    case 128: return &v128;
    case 216: return &v216;
  }
  return nullptr;
}
}  // namespace spx
