// Instantiation unit: the fused y pass for float, three groups per column (up to 1024 points).
#include "gf_ystage_impl.hpp"
namespace gf {
void ystage_long_f(int n, const K3Args<float>& c, const K1Args<float>& a, hipStream_t s);
template <> void launch_ystage<float>(int n, int groups, const K3Args<float>& c, const K1Args<float>& a, hipStream_t s) {
  if (groups == 1) { ystage_long_f(n, c, a, s); return; }
  switch (n) {
    case 32: ystage_n<float, 32, 3>(c, a, s); break;
    case 64: ystage_n<float, 64, 3>(c, a, s); break;
    case 128: ystage_n<float, 128, 3>(c, a, s); break;
    case 256: ystage_n<float, 256, 3>(c, a, s); break;
    case 512: ystage_n<float, 512, 3>(c, a, s); break;
    case 1024: ystage_n<float, 1024, 3>(c, a, s); break;
    default: break;
  }
}
}  // namespace gf
