// Instances of the two-pass volume kernels (volume.h).
#include "volume.h"

namespace spx {
const VolOps* vol_ops_0(int L) {
  static const VolOps v64 = vol_ops_of<64>();
  static const VolOps v72 = vol_ops_of<72>();
  static const VolOps v256 = vol_ops_of<256>();
  switch (L) {
    case 64: return &v64;
    case 72: return &v72;
    case 256: return &v256;
  }
  return nullptr;
}
}  // namespace spx
