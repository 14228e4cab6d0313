// Instantiation unit: the fused y pass of double problems whose columns are not a power of two long.
#include "gf_ylayers_impl.hpp"
namespace gf {
void ylayers_ragged_d(int ny, const K3Args<double>& c, const K1Args<double>& a, hipStream_t s) {
  switch (pow2_ceil(ny)) {
    case 32: ylayers_l<double, 32, true>(c, a, s); break;
    case 64: ylayers_l<double, 64, true>(c, a, s); break;
    case 128: ylayers_l<double, 128, true>(c, a, s); break;
    case 256: ylayers_l<double, 256, true>(c, a, s); break;
    default: break;
  }
}
}  // namespace gf
