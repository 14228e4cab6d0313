// Instantiation unit: the fused y pass of multi-layer double problems, power-of-two columns.
#include "gf_ylayers_impl.hpp"
namespace gf {
void ylayers_ragged_d(int ny, const K3Args<double>& c, const K1Args<double>& a, hipStream_t s);
template <> void launch_ylayers<double>(int ny, const K3Args<double>& c, const K1Args<double>& a, hipStream_t s) {
  if (!is_pow2(ny)) { ylayers_ragged_d(ny, c, a, s); return; }
  switch (pow2_ceil(ny)) {
    case 32: ylayers_l<double, 32, false>(c, a, s); break;
    case 64: ylayers_l<double, 64, false>(c, a, s); break;
    case 128: ylayers_l<double, 128, false>(c, a, s); break;
    case 256: ylayers_l<double, 256, false>(c, a, s); break;
    case 512: ylayers_l<double, 512, false>(c, a, s); break;
    default: break;
  }
}
}  // namespace gf
