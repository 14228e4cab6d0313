// Batched ensembles in two launches per stage: the x pass and the fused y pass of every member, over a
// flat table of (instance, block) entries as the three-launch form walks it.
//
// Every transform is held by one wave, so none of its exchanges needs a barrier.  NG = 3, 192-thread
// workgroups: the forms a single small problem runs (k2_group_body, ystage_body with three groups), 4 points
// per thread up to 256 and 8 at 512, for ensembles that leave the GPU waiting on latency.  NG = 1, 64-thread
// workgroups: one wave per entry runs its five transforms in a row at 8 points per thread (an exchange
// fewer), for ensembles that fill the GPU, where idle groups cost more than they save.  The three-launch form ran each entry on 256 threads with barriers at every exchange and wrote the
// state out between K3 and K1; it still serves ensembles with a one-layer MultiLayerQG member (its
// drag reads a state that this form does not store), per-class timing and the persistent form.
#include "gf_ystage_impl.hpp"

namespace gf {

constexpr int BATCH2_TW = 128;
template <int N, int NG> struct Batch2 {
  static constexpr int P = NG == 1 || N >= 512 ? 8 : 4;
  static constexpr int CPW = k3_single_column(N, P) ? 1 : 2;
  static_assert(K2P<N, P>::GT == 64 && YS<N, P, 3, CPW>::GT == 64 && YS<N, P, 1, CPW>::GT == 64, "one wave per group");
  static_assert(TwPlan<N, P>::size() <= BATCH2_TW, "twiddle table");
};
// LDS slots of members up to nmax
template <typename T, int N, int NG> constexpr int batch2_slots() {
  constexpr int x = NG * K2P<N, Batch2<N, NG>::P>::G * LdsN<N>::value, y = YLds<T, N, Batch2<N, NG>::P, NG, Batch2<N, NG>::CPW>::value;
  return x > y ? x : y;
}
template <typename T, int NG> size_t batch2_lds(int nmax) {
  const int n[5] = {32, 64, 128, 256, 512};
  const int s[5] = {batch2_slots<T, 32, NG>(), batch2_slots<T, 64, NG>(), batch2_slots<T, 128, NG>(), batch2_slots<T, 256, NG>(),
                    batch2_slots<T, 512, NG>()};
  int m = 0;
  for (int i = 0; i < 5; ++i) if (n[i] <= nmax && s[i] > m) m = s[i];
  return sizeof(cplx<T>) * (size_t)m;
}

template <typename T, int N, int NG, int MODE>
__device__ __forceinline__ void batch2_xn(const BatchItem<T>& it, int blk, cplx<T>* lds, cplx<T>* tw) {
  constexpr int P = Batch2<N, NG>::P;
  if constexpr (NG == 3) {
    k2_group_body<T, N, P, MODE>(it.k2, blk, 0, lds, tw);
  } else {
    load_twiddles<T, N, P>(tw, it.k2.tw);
    xbarrier<X_WAVE>();
    k2_body<T, N, P, K2P<N, P>::G, MODE, 1, X_WAVE>(it.k2, blk, lds, tw);
  }
}
template <typename T, int N, int NG, bool PLAIN>
__device__ __forceinline__ void batch2_x(const BatchItem<T>& it, int blk, cplx<T>* lds, cplx<T>* tw) {
  if (!PLAIN && it.k2.mode == K2_ADVECT_FULL) {
    if constexpr (!PLAIN) batch2_xn<T, N, NG, K2_ADVECT_FULL>(it, blk, lds, tw);
  } else if (!PLAIN && it.k2.mode == K2_ADVECT_Y) {
    if constexpr (!PLAIN) batch2_xn<T, N, NG, K2_ADVECT_Y>(it, blk, lds, tw);
  } else {
    batch2_xn<T, N, NG, K2_ADVECT>(it, blk, lds, tw);
  }
}
template <typename T, int N, int NG>
__device__ __forceinline__ void batch2_y(const BatchItem<T>& it, int blk, int mode, cplx<T>* lds, cplx<T>* tw) {
  using B = Batch2<N, NG>;
  constexpr bool AHEAD = NG == 3 && N < 512;
  if (it.k1.model == M_TWODNS) ystage_body<T, N, B::P, NG, B::CPW, M_TWODNS, -1, AHEAD>(it.k3, it.k1, blk, mode, lds, tw);
  else ystage_body<T, N, B::P, NG, B::CPW, M_SLQG, -1, AHEAD>(it.k3, it.k1, blk, mode, lds, tw);
}

template <typename T, int NG, bool PLAIN>
__global__ __launch_bounds__((NG * 64)) __attribute__((amdgpu_waves_per_eu(PLAIN ? 4 : 2)))
void batch2_x_kernel(const BatchItem<T>* __restrict__ items, const BatchWork* __restrict__ work) {
  extern __shared__ __align__(16) char dyn[];
  __shared__ cplx<T> tw[BATCH2_TW];
  cplx<T>* lds = reinterpret_cast<cplx<T>*>(dyn);
  const BatchWork w = work[blockIdx.x];
  const BatchItem<T>& it = items[w.item];
  switch (it.n) {
    case 32: batch2_x<T, 32, NG, PLAIN>(it, w.blk, lds, tw); break;
    case 64: batch2_x<T, 64, NG, PLAIN>(it, w.blk, lds, tw); break;
    case 128: batch2_x<T, 128, NG, PLAIN>(it, w.blk, lds, tw); break;
    case 256: batch2_x<T, 256, NG, PLAIN>(it, w.blk, lds, tw); break;
    case 512: batch2_x<T, 512, NG, PLAIN>(it, w.blk, lds, tw); break;
    default: break;
  }
}
template <typename T, int NG>
__global__ __launch_bounds__((NG * 64)) __attribute__((amdgpu_waves_per_eu(3)))
void batch2_y_kernel(const BatchItem<T>* __restrict__ items, const BatchWork* __restrict__ work, int mode) {
  extern __shared__ __align__(16) char dyn[];
  __shared__ cplx<T> tw[BATCH2_TW];
  cplx<T>* lds = reinterpret_cast<cplx<T>*>(dyn);
  const BatchWork w = work[blockIdx.x];
  const BatchItem<T>& it = items[w.item];
  switch (it.n) {
    case 32: batch2_y<T, 32, NG>(it, w.blk, mode, lds, tw); break;
    case 64: batch2_y<T, 64, NG>(it, w.blk, mode, lds, tw); break;
    case 128: batch2_y<T, 128, NG>(it, w.blk, mode, lds, tw); break;
    case 256: batch2_y<T, 256, NG>(it, w.blk, mode, lds, tw); break;
    case 512: batch2_y<T, 512, NG>(it, w.blk, mode, lds, tw); break;
    default: break;
  }
}

template <typename T>
void launch_batch_x(const BatchItem<T>* items, const BatchWork* work, int nwork, int nmax, int groups, int plain, hipStream_t s) {
  if (nwork <= 0) return;
  const dim3 grid(nwork), blk(groups == 3 ? 192 : 64);
  const size_t sh = groups == 3 ? batch2_lds<T, 3>(nmax) : batch2_lds<T, 1>(nmax);
  if (groups == 3) {
    if (plain) hipLaunchKernelGGL((batch2_x_kernel<T, 3, true>), grid, blk, sh, s, items, work);
    else hipLaunchKernelGGL((batch2_x_kernel<T, 3, false>), grid, blk, sh, s, items, work);
  } else {
    if (plain) hipLaunchKernelGGL((batch2_x_kernel<T, 1, true>), grid, blk, sh, s, items, work);
    else hipLaunchKernelGGL((batch2_x_kernel<T, 1, false>), grid, blk, sh, s, items, work);
  }
}
template <typename T>
void launch_batch_y(const BatchItem<T>* items, const BatchWork* work, int nwork, int nmax, int groups, int mode, hipStream_t s) {
  if (nwork <= 0) return;
  const size_t sh = groups == 3 ? batch2_lds<T, 3>(nmax) : batch2_lds<T, 1>(nmax);
  if (groups == 3) hipLaunchKernelGGL((batch2_y_kernel<T, 3>), dim3(nwork), dim3(192), sh, s, items, work, mode);
  else hipLaunchKernelGGL((batch2_y_kernel<T, 1>), dim3(nwork), dim3(64), sh, s, items, work, mode);
}

}  // namespace gf
