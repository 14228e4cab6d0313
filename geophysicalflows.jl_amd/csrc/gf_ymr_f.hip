// Instantiation unit: the fused y pass of float problems whose columns are not a power of two long.
#include "gf_ylayers_impl.hpp"
namespace gf {
void ylayers_ragged_f(int ny, const K3Args<float>& c, const K1Args<float>& a, hipStream_t s) {
  switch (pow2_ceil(ny)) {
    case 32: ylayers_l<float, 32, true>(c, a, s); break;
    case 64: ylayers_l<float, 64, true>(c, a, s); break;
    case 128: ylayers_l<float, 128, true>(c, a, s); break;
    case 256: ylayers_l<float, 256, true>(c, a, s); break;
    default: break;
  }
}
}  // namespace gf
