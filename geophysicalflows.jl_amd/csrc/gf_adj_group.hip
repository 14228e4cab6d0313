// The adjoint kernels (gf_adjoint_impl.hpp) of grids up to 512^2, a wave per transform, in two launches per stage:
// KA2 with its five inverse and then its three forward transforms side by side, and KA3 of a stage with
// KA1 of the next one on the same columns.
//
// One gradient leaves the GPU waiting on latency: KA2 ran eight transforms in a row and KA1, KA3 eight more,
// with barriers at every exchange and the co-states through HBM in between.  Here a transform is one wave's (no
// barriers), a row pair or column takes two in a row, and the co-state that the next KA1 reads stays in
// LDS.  512^2 FP64 per stage: KA1 9.5 + KA2 12.9 + KA3 12.9 us -> 14.7 + 8.9.
#include "gf_kernels_impl.hpp"

namespace gf {

template <typename T> __device__ __forceinline__ T herm_weight(const Geo<T>& g, int kr) {
  return (kr == 0 || 2 * kr == g.nx) ? (T)1 : (T)2;
}

template <int N> struct AG {
  static constexpr int P = ylayers_p(N), TPT = N / P;
  static constexpr int CPW = k3_single_column(N, P) ? 1 : 2;
  static constexpr int GC = CPW == 2 ? GY<N, P>::G : 1;    // column pairs (columns) per wave
  static constexpr int GR = K2P<N, P>::G;                  // row pairs per wave
  static_assert(CPW * GC * TPT == 64 && GR * TPT == 64, "a group is one wave");
};

// ---- KA2: wave f transforms field f (u, v, zeta, pA, pB); waves 0, 1, 2 the products zeta pA, zeta pB, u pA + v pB
template <typename T, int NX>
__global__ __launch_bounds__(320)
void ka2_group_kernel(const AdjK2Args<T> a) {
  using A = AG<NX>;
  constexpr int P = A::P, TPT = A::TPT, G = A::GR, PG = XPad<T>::G;
  constexpr int MAXI = (NX / 2 + 1 + TPT - 1) / TPT;
  constexpr int QH = P / 2 + 1;
  __shared__ cplx<T> lds[5 * G * LdsN<NX>::value];
  __shared__ cplx<T> tw[TwPlan<NX, P>::size()];
  const Geo<T>& g = a.g;
  const int ny = g.ny;
  const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int t = (int)threadIdx.x % TPT, slot = ((int)threadIdx.x % 64) / TPT;
  const int rp = xcd_block(blockIdx.x, gridDim.x) * G + slot;
  const bool active = rp < ny / 2;
  const int y0 = 2 * rp;
  auto buffer = [&](int f) { return lds + (f * G + slot) * LdsN<NX>::value; };
  cplx<T>* L = buffer(grp);
  cplx<T> w[1][P];
  {
    // the Hermitian half k > NX/2 comes from the mirror's lane (k2_body)
    const cplx<T>* f = a.in + (long)grp * a.fstride;
    cplx<T> A0[QH], B0[QH];
#pragma unroll
    for (int q = 0; q < QH; ++q) {
      const int k = t + TPT * q;
      A0[q] = herm_load<T, NX>(f, k, y0, ny, a.kin, active && k <= NX / 2);
      B0[q] = herm_load<T, NX>(f, k, y0 + 1, ny, a.kin, active && k <= NX / 2);
    }
    load_twiddles<T, NX, P>(tw, a.tw);
#pragma unroll
    for (int q = 0; q < QH; ++q) {
      const int k = t + TPT * q;
      if (k > NX / 2) continue;
      w[0][q] = mk(A0[q].re - B0[q].im, -(A0[q].im + B0[q].re));
      if (k > 0 && k < NX / 2) L[padg<PG>(NX - k)] = mk(A0[q].re + B0[q].im, A0[q].im - B0[q].re);
    }
    lds_barrier();
#pragma unroll
    for (int q = 0; q < P; ++q) {
      if (TPT * q + TPT - 1 <= NX / 2) continue;
      const int k = t + TPT * q;
      if (k <= NX / 2) continue;
      w[0][q] = L[padg<PG>(k)];
    }
    xbarrier<X_WAVE>();
  }
  fft_forward<T, NX, P, 1, false, X_WAVE>(w, L, t, tw);   // row y0 = Re, row y0 + 1 = -Im
  const int off = padg<PG>(t);
#pragma unroll
  for (int q = 0; q < P; ++q) L[off + padg<PG>(TPT * q)] = conj(w[0][q]);
  lds_barrier();
  if (grp < 3) {
    const cplx<T>*u = buffer(0) + off, *v = buffer(1) + off, *z = buffer(2) + off, *pa = buffer(3) + off, *pb = buffer(4) + off;
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int s = padg<PG>(TPT * q);
      if (grp < 2) {
        const cplx<T> x = z[s], p = grp == 0 ? pa[s] : pb[s];
        w[0][q] = mk(x.re * p.re, x.im * p.im);
      } else {
        const cplx<T> x = u[s], p = pa[s], y = v[s], r = pb[s];
        w[0][q] = mk(x.re * p.re + y.re * r.re, x.im * p.im + y.im * r.im);
      }
    }
  }
  lds_barrier();                                       // the rows are read: the buffers are free
  if (grp >= 3) return;
  fft_forward<T, NX, P, 1, false, X_WAVE>(w, L, t, tw);
  const MirrorSlots<NX, TPT, PG> ms(t);
#pragma unroll
  for (int q = 0; q < P; ++q) L[ms.k(q)] = w[0][q];
  xbarrier<X_WAVE>();
  if (!active) return;
  cplx<T>* o = a.out + (long)grp * a.ostride;
#pragma unroll
  for (int i = 0; i < MAXI; ++i) {
    const int kr = t + i * TPT;
    if (kr < a.kout) {
      const cplx<T> Wk = L[ms.k(i)], Wm = L[ms.m(i)];
      at(o, boff32(kr, y0, ny)) = split_row(Wk, Wm, 0);
      at(o, boff32(kr, y0 + 1, ny)) = split_row(Wk, Wm, 1);
    }
  }
}

// ---- KA3 of the stage k, then KA1 (a) of the next: mode 0 KA1 alone, 1 both, 2 KA3 alone
template <typename T, int NY>
__global__ __launch_bounds__(320)
void kay_kernel(const AdjK3Args<T> k, const AdjK1Args<T> a, int mode) {
  using A = AG<NY>;
  constexpr int P = A::P, TPT = A::TPT, G = A::GC, CPW = A::CPW, PG = XPad<T>::G;
  constexpr int BUF = CPW == 2 ? G * PairLds<T, NY>::value : LdsN<NY>::value;
  constexpr int QN = (P + 4) / 5;
  __shared__ cplx<T> lds[5 * BUF];
  __shared__ cplx<T> tw[TwPlan<NY, P>::size()];
  __shared__ T part[5];
  const Geo<T>& g = k.g;
  const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  int t, kr, col;
  if constexpr (CPW == 2) {
    const YMap<TPT> m((int)threadIdx.x % 64);
    t = m.t;
    kr = 2 * (G == 1 ? pair_of_block(blockIdx.x) : (int)blockIdx.x * G + m.slot) + m.c;
    col = (int)(col_buffer<T, NY>(lds, m.slot, m.c) - lds);
  } else {
    t = (int)threadIdx.x % 64;
    kr = single_column(blockIdx.x);
    col = 0;
  }
  cplx<T>* L = lds + grp * BUF + col;
  const int off = padg<PG>(t);
  const T kv = krwave(g, kr);
  const bool active = kr < g.kmax && kr < k.ncols;
  const int krl = active ? kr : 0;
  cplx<T> w[1][P], sv[P];
  if (mode != 2 && grp < 3) {
    // the next stage's calcN input, rebuilt from the tape (ka1_body's stage_state), under way early
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int l = t + TPT * q;
      const uint32_t ix = boff32(krl, l, NY);
      const cplx<T> s0 = at(a.s0, ix);
      cplx<T> v = s0;
      if (a.stage != 1) {
        const T E2 = at(a.E2, ix), Z = at(a.Z, ix);
        const cplx<T> nb = at(a.stage == 3 ? a.N2 : a.N1, ix);
        v = rfma(E2, s0, rmul(Z, nb));
        if (a.stage == 4) {
          const cplx<T> n3 = at(a.N3, ix);
          v = rfma(E2, v, rmul(Z, mk((T)2 * n3.re - nb.re, (T)2 * n3.im - nb.im)));
        }
      }
      sv[q] = active && kept_l(g, l) ? v : czero<T>();
    }
  }
  load_twiddles<T, NY, P>(tw, k.tw);
  cplx<T>* S = lds + 3 * BUF + col;
  if (mode == 0) {
#pragma unroll
    for (int i = 0; i < QN; ++i) {
      const int q = grp + 5 * i, l = t + TPT * q;
      if (q >= P) continue;
      const cplx<T> x = at(a.x, boff32(krl, l, NY));
      S[padg<PG>(l)] = active && kept_l(g, l) ? x : czero<T>();
    }
    lds_barrier();
  } else {
    const cplx<T>* f = k.in + (long)(grp < 3 ? grp : 0) * k.fstride;
#pragma unroll
    for (int q = 0; q < P; ++q) w[0][q] = at(f, boff32(krl, t + TPT * q, NY));
    lds_barrier();                                     // the twiddles
    fft_forward<T, NY, P, 1, false, X_WAVE>(w, L, t, tw);
    if (grp < 3) {
#pragma unroll
      for (int q = 0; q < P; ++q) L[off + padg<PG>(TPT * q)] = w[0][q];
    }
    lds_barrier();
    // lambda_s and the adjoint stage arithmetic (ka3_body) of this thread's rows; x: the co-state of the
    // next stage's N, which its KA1 reads (only what later stages read is stored)
    const cplx<T>* F = lds + col;
    const T wk = herm_weight(g, kr);
    T nu = 0;
#pragma unroll
    for (int i = 0; i < QN; ++i) {
      const int q = grp + 5 * i, l = t + TPT * q;
      if (q >= P) continue;
      const int s = padg<PG>(l);
      cplx<T> x = czero<T>();
      if (active && kept_l(g, l)) {
        const T lv = lwave(g, l), iK = inv_k2(kr, l, kv, lv);
        const cplx<T> f0 = F[s], f1 = F[BUF + s], f2 = F[2 * BUF + s];
        const T cl = lv * iK, ck = kv * iK;
        // F(u pA + v pB) - i l/|k|^2 F(zeta pA) + i kr/|k|^2 F(zeta pB)
        const cplx<T> acc = f2 + mk(cl * f0.im - ck * f1.im, ck * f1.re - cl * f0.re);
        const cplx<T> tv = rmul(wk, acc);
        const uint32_t ix = boff32(kr, l, NY);
        const T E2 = at(k.E2, ix), Z = at(k.Z, ix);
        auto re_dot = [](cplx<T> p, cplx<T> r) { return p.re * r.re + p.im * r.im; };
        if (k.stage == 4) {
          const cplx<T> lam = at(k.lam, ix);
          const T Al = at(k.Al, ix), Be = at(k.Be, ix);
          at(k.l1, ix) = rmul(E2, tv);
          x = rfma((T)2 * Be, lam, rmul((T)2 * Z, tv));           // lambda of N3
          at(k.lN1, ix) = rfma(Al, lam, rmul(-Z, tv));
          if (k.nu_part != nullptr) {
            const cplx<T> s0 = at(k.s0, ix), N1 = at(k.N1, ix), N2 = at(k.N2, ix), N3 = at(k.N3, ix), N4 = at(k.N4, ix);
            const cplx<T> s1 = rfma(E2, s0, rmul(Z, N1));
            const cplx<T> d1 = rfma(at(k.dE, ix), s0, rfma(at(k.dA, ix), N1, rfma((T)2 * at(k.dB, ix), N2 + N3, rmul(at(k.dG, ix), N4))));
            const cplx<T> d3 = rfma(at(k.dE2, ix), s1, rmul(at(k.dZ, ix), mk((T)2 * N3.re - N1.re, (T)2 * N3.im - N1.im)));
            nu += re_dot(lam, d1) + re_dot(tv, d3);
          }
        } else if (k.stage == 3) {
          const cplx<T> lam = at(k.lam, ix);
          const T E = at(k.E, ix), Be = at(k.Be, ix);
          at(k.l0, ix) = rfma(E, lam, rmul(E2, tv));
          x = rfma((T)2 * Be, lam, rmul(Z, tv));                  // lambda of N2
          if (k.nu_part != nullptr) nu += re_dot(tv, rfma(at(k.dE2, ix), at(k.s0, ix), rmul(at(k.dZ, ix), at(k.N2, ix))));
        } else if (k.stage == 2) {
          const cplx<T> l1 = at(k.l1, ix) + tv;
          at(k.l0, ix) = rfma(E2, l1, at(k.l0, ix));
          x = rfma(Z, l1, at(k.lN1, ix));                         // lambda of N1
          if (k.nu_part != nullptr) nu += re_dot(l1, rfma(at(k.dE2, ix), at(k.s0, ix), rmul(at(k.dZ, ix), at(k.N1, ix))));
        } else {
          x = at(k.l0, ix) + tv;                                  // lambda of the step's input
          at(k.lam, ix) = x;
        }
      }
      S[s] = x;
    }
    if (k.nu_part != nullptr && k.stage >= 2) {
      // workgroup sum of the nu terms in a fixed order: lanes, then waves
#pragma unroll
      for (int s = 32; s > 0; s >>= 1) nu += __shfl_down(nu, s, 64);
      if ((threadIdx.x & 63) == 0) part[grp] = nu;
    }
    lds_barrier();
    if (k.nu_part != nullptr && k.stage >= 2 && threadIdx.x == 0)
      k.nu_part[blockIdx.x] += (((part[0] + part[1]) + part[2]) + part[3]) + part[4];
    if (mode == 2) return;
  }

  // wave f: field f of the next stage, u, v, zeta of its calcN input or pA, pB of its co-state
  if (grp >= 3) {
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int l = t + TPT * q;
      cplx<T> x = S[off + padg<PG>(TPT * q)];
      if (a.lamc != nullptr) x = rmul(at(a.lamc, boff32(krl, l, NY)), x);
      sv[q] = x;
    }
  }
  lds_barrier();                                       // the co-state is read: the buffers are free
  const T nrm = g.inv_norm, wi = (T)1 / herm_weight(g, kr);
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int l = t + TPT * q;
    const T lv = lwave(g, l);
    cplx<T> r;
    if (grp < 3) {
      const T iK = inv_k2(kr, l, kv, lv);
      if (grp == 0) { const T c = lv * iK; r = mk(-c * sv[q].im, c * sv[q].re); }         // u: i l s/|k|^2
      else if (grp == 1) { const T c = kv * iK; r = mk(c * sv[q].im, -c * sv[q].re); }    // v: -i kr s/|k|^2
      else r = sv[q];
    } else {
      const T c = (grp == 3 ? kv : lv) * wi;                                              // i kr/w, i l/w
      r = mk(-c * sv[q].im, c * sv[q].re);
    }
    w[0][q] = mk(r.re * nrm, -(r.im * nrm));
  }
  fft_forward<T, NY, P, 1, false, X_WAVE>(w, L, t, tw);
  if (active) {
    cplx<T>* o = a.out + (long)grp * a.fstride;
#pragma unroll
    for (int q = 0; q < P; ++q) at(o, boff32(kr, t + TPT * q, NY)) = conj(w[0][q]);
  }
}

template <int N> static int kay_blocks(int ncols) { return AG<N>::CPW == 1 ? column_blocks(ncols) : pair_blocks(ncols, AG<N>::GC); }
bool adj_group_built(int n) { return n >= 32 && n <= 512; }
int adj_group_blocks(int n, int ncols) {
  switch (n) {
    case 32: return kay_blocks<32>(ncols);
    case 64: return kay_blocks<64>(ncols);
    case 128: return kay_blocks<128>(ncols);
    case 256: return kay_blocks<256>(ncols);
    default: return kay_blocks<512>(ncols);
  }
}
template <int N> static void adj_go(const AdjK1Args<double>* a, const AdjK2Args<double>* b, const AdjK3Args<double>* k, int mode, hipStream_t s) {
  if (b) {
    const int nblk = (b->g.ny / 2 + AG<N>::GR - 1) / AG<N>::GR;
    hipLaunchKernelGGL((ka2_group_kernel<double, N>), dim3(nblk), dim3(320), 0, s, *b);
    return;
  }
  const int nblk = kay_blocks<N>(k->ncols);
  if (nblk > 0) hipLaunchKernelGGL((kay_kernel<double, N>), dim3(nblk), dim3(320), 0, s, *k, *a, mode);
}
static void adj_dispatch(int n, const AdjK1Args<double>* a, const AdjK2Args<double>* b, const AdjK3Args<double>* k, int mode, hipStream_t s) {
  switch (n) {
    case 32: adj_go<32>(a, b, k, mode, s); break;
    case 64: adj_go<64>(a, b, k, mode, s); break;
    case 128: adj_go<128>(a, b, k, mode, s); break;
    case 256: adj_go<256>(a, b, k, mode, s); break;
    case 512: adj_go<512>(a, b, k, mode, s); break;
    default: break;
  }
}
void launch_adj_x(int n, const AdjK2Args<double>& b, hipStream_t s) { adj_dispatch(n, nullptr, &b, nullptr, 0, s); }
void launch_adj_y(int n, const AdjK3Args<double>& k, const AdjK1Args<double>& a, int mode, hipStream_t s) { adj_dispatch(n, &a, nullptr, &k, mode, s); }

}  // namespace gf
