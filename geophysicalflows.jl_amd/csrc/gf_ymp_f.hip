// Instantiation unit: the fused y pass of multi-layer float problems, power-of-two columns.
#include "gf_ylayers_impl.hpp"
namespace gf {
void ylayers_ragged_f(int ny, const K3Args<float>& c, const K1Args<float>& a, hipStream_t s);
template <> void launch_ylayers<float>(int ny, const K3Args<float>& c, const K1Args<float>& a, hipStream_t s) {
  if (!is_pow2(ny)) { ylayers_ragged_f(ny, c, a, s); return; }
  switch (pow2_ceil(ny)) {
    case 32: ylayers_l<float, 32, false>(c, a, s); break;
    case 64: ylayers_l<float, 64, false>(c, a, s); break;
    case 128: ylayers_l<float, 128, false>(c, a, s); break;
    case 256: ylayers_l<float, 256, false>(c, a, s); break;
    case 512: ylayers_l<float, 512, false>(c, a, s); break;
    default: break;
  }
}
}  // namespace gf
