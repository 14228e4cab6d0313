// Instantiation unit: the two-launch stages of float ensembles.
#include "gf_batch_y_impl.hpp"
namespace gf {
template void launch_batch_x<float>(const BatchItem<float>*, const BatchWork*, int, int, int, int, hipStream_t);
template void launch_batch_y<float>(const BatchItem<float>*, const BatchWork*, int, int, int, int, hipStream_t);
}  // namespace gf
