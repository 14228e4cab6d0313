// Instantiation unit: the two-launch stages of double ensembles.
#include "gf_batch_y_impl.hpp"
namespace gf {
template void launch_batch_x<double>(const BatchItem<double>*, const BatchWork*, int, int, int, int, hipStream_t);
template void launch_batch_y<double>(const BatchItem<double>*, const BatchWork*, int, int, int, int, hipStream_t);
template <int N, int NG> static int blocks2(int y, int count) {
  using B = Batch2<N, NG>;
  if (!y) return (count / 2 + K2P<N, B::P>::G - 1) / K2P<N, B::P>::G;
  return B::CPW == 1 ? column_blocks(count) : pair_blocks(count, YS<N, B::P, NG, B::CPW>::G);
}
template <int NG> static int blocks2_n(int y, int n, int count) {
  switch (n) {
    case 32: return blocks2<32, NG>(y, count);
    case 64: return blocks2<64, NG>(y, count);
    case 128: return blocks2<128, NG>(y, count);
    case 256: return blocks2<256, NG>(y, count);
    default: return blocks2<512, NG>(y, count);
  }
}
int batch2_blocks(int y, int n, int count, int groups) {
  return groups == 3 ? blocks2_n<3>(y, n, count) : blocks2_n<1>(y, n, count);
}
}  // namespace gf
