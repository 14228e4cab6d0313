// Instantiation unit: the fused y pass for double, one group per column (from 1024 points).
#include "gf_ystage_impl.hpp"
namespace gf {
void ystage_long_d(int n, const K3Args<double>& c, const K1Args<double>& a, hipStream_t s) {
  switch (n) {
    case 1024: ystage_n<double, 1024, 1>(c, a, s); break;
    case 2048: ystage_n<double, 2048, 1>(c, a, s); break;
    case 4096: ystage_n<double, 4096, 1>(c, a, s); break;
    default: break;
  }
}
}  // namespace gf
