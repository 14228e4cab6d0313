// Instantiation unit: the fused y pass for double, three groups per column (up to 1024 points).
#include "gf_ystage_impl.hpp"
namespace gf {
void ystage_long_d(int n, const K3Args<double>& c, const K1Args<double>& a, hipStream_t s);
template <> void launch_ystage<double>(int n, int groups, const K3Args<double>& c, const K1Args<double>& a, hipStream_t s) {
  if (groups == 1) { ystage_long_d(n, c, a, s); return; }
  switch (n) {
    case 32: ystage_n<double, 32, 3>(c, a, s); break;
    case 64: ystage_n<double, 64, 3>(c, a, s); break;
    case 128: ystage_n<double, 128, 3>(c, a, s); break;
    case 256: ystage_n<double, 256, 3>(c, a, s); break;
    case 512: ystage_n<double, 512, 3>(c, a, s); break;
    case 1024: ystage_n<double, 1024, 3>(c, a, s); break;
    default: break;
  }
}
}  // namespace gf
