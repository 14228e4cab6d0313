// Instantiation unit: the fused y pass for float, one group per column (from 1024 points).
#include "gf_ystage_impl.hpp"
namespace gf {
void ystage_long_f(int n, const K3Args<float>& c, const K1Args<float>& a, hipStream_t s) {
  switch (n) {
    case 1024: ystage_n<float, 1024, 1>(c, a, s); break;
    case 2048: ystage_n<float, 2048, 1>(c, a, s); break;
    case 4096: ystage_n<float, 4096, 1>(c, a, s); break;
    default: break;
  }
}
}  // namespace gf
