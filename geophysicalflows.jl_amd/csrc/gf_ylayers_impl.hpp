// The fused y pass (gf_ystage_impl.hpp) of multi-layer problems, and of columns whose length is not a power
// of two: K3 of one stage and K1 of the next for all layers of a column in one workgroup.
//
// Each of the 2 NL flux transforms and then each of the 3 NL field transforms has a wave of its own, so a
// column takes two transforms in a row where K3 and K1 took five per layer; the waves meet in LDS, where
// also the layers do for psih = S^-1 q.  3 NL waves: NL = 1 (columns that are not a power of two; the
// others have ystage_kernel) to 5; up to 512 points, 8 per thread at 512 and 4 below, one column or
// column pairs per wave.  More layers or points run K3 and K1.
// FP64 per launch, K3 + K1 -> fused: MultiLayerQG 512^2 x 3 11.9 + 12.8 -> 16.3 us, 128x126 x 2 12.9 + 11.4 -> 13.4.
#include "gf_kernels_impl.hpp"

namespace gf {

template <typename T, int NY, int P, int NL, int CPW, bool GEN> struct YL {
  static constexpr int TPT = NY / P;
  static constexpr int G = CPW == 2 ? GY<NY, P>::G : 1;
  static constexpr int NG = 3 * NL;
  static constexpr int NB = YN<NY, GEN>::value;        // points of a column's buffer
  static constexpr int BUF = CPW == 2 ? G * PairLds<T, NB>::value : LdsN<NB>::value;
  static constexpr int QN = (P + 2) / 3;               // modes a thread steps: NL P over 3 NL groups
  static constexpr bool AHEAD = NL <= 2 || (NL == 3 && P == 4);   // their reads issued before the transforms (registers)
  static_assert(CPW * G * TPT == 64, "a group is one wave");
};

template <typename T, int NY, int P, int NL, int CPW, int MODEL, bool GEN>
__global__ __launch_bounds__((64 * 3 * NL))
void ylayers_kernel(const K3Args<T> c, const K1Args<T> a) {
  using Y = YL<T, NY, P, NL, CPW, GEN>;
  constexpr int TPT = Y::TPT, G = Y::G, PG = XPad<T>::G, BUF = Y::BUF, NG = Y::NG;
  __shared__ cplx<T> lds[NG * BUF];
  __shared__ cplx<T> tw[YTw<NY, P, GEN>::size];
  const Geo<T>& g = c.g;
  const int ny = ycol<NY, GEN>(g);
  const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  int t, kr, col;
  if constexpr (CPW == 2) {
    const YMap<TPT> m((int)threadIdx.x % 64);
    t = m.t;
    kr = 2 * (G == 1 ? pair_of_block(blockIdx.x) : (int)blockIdx.x * G + m.slot) + m.c;
    col = (int)(col_buffer<T, Y::NB>(lds, m.slot, m.c) - lds);
  } else {
    t = (int)threadIdx.x % 64;
    kr = single_column(blockIdx.x);
    col = 0;
  }
  cplx<T>* L = lds + grp * BUF + col;
  const T kv = krwave(g, kr);
  const bool active = kr < c.ncols && kr < g.nkr;
  const int krl = active ? kr : 0;
  const int epi = c.epi;
  // (lanes past the column's end read its first row and drop what they make of it)
  auto safe = [&](int l) { return in_col<GEN>(l, ny) ? l : 0; };

  cplx<T> w[1][P];
  {
    const cplx<T>* f = c.in + (long)(grp < 2 * NL ? grp : 0) * c.fstride;
#pragma unroll
    for (int q = 0; q < P; ++q) w[0][q] = at(f, boff32(krl, safe(t + TPT * q), ny));
  }
  load_y_twiddles<T, NY, P, GEN>(tw, c.tw, ny);
  // this thread's modes: number i is row t + TPT q of layer jl, (jl, q) counted through grp + NG i
  auto mine = [&](int i) { return grp + NG * i < NL * P; };
  auto layer = [&](int i) { return (grp + NG * i) / P; };
  auto row = [&](int i) { return t + TPT * ((grp + NG * i) % P); };
  auto point = [&](int i) {
    const bool m = mine(i);
    return StagePoint<T>(c, krl, m ? safe(row(i)) : safe(t), ny, (uint32_t)((m ? layer(i) : 0) * g.lstride));
  };
  StageIn<T> in[Y::AHEAD ? Y::QN : 1];
  if constexpr (Y::AHEAD) {
#pragma unroll
    for (int i = 0; i < Y::QN; ++i) in[i] = stage_load<T>(c, epi, point(i));
  }
  // ring forcing: this thread's terms, read back by it in the stage; a slice of the box per layer
  if (c.sqrt_spec != nullptr && active && kr <= c.fkx) {
    const int64_t fstep = c.fstep_dev != nullptr ? c.fstep_dev[0] : c.fstep;
    for (int i = 0; i < Y::QN; ++i) {
      const int l = row(i);
      if (mine(i) && in_col<GEN>(l, ny) && (l <= c.fky || l >= ny - c.fky)) {
        const T sp = at(c.sqrt_spec, boff32(kr, l, ny));
        if (sp != (T)0) {
          const cplx<T> xi = complex_normal<T>(c.seed, fstep, (uint32_t)(l * g.nkr + kr), (uint32_t)c.instance);
          c.noise[(long)layer(i) * (c.fkx + 1) * c.nbl + kr * c.nbl + ring_box_row(l, ny, c.fky, c.nbl)] =
              mk((xi.re * sp) / c.sqrt_dt, (xi.im * sp) / c.sqrt_dt);
        }
      }
    }
  }
  lds_barrier();                                       // the twiddles
  y_transform<T, NY, P, false, GEN, X_WAVE>(w, L, t, tw, ny);

  // flux f of layer jl crosses groups in buffer 2 jl + f, the new modes of layer jl in buffer 2 NL + jl
  const int off = padg<PG>(t);
  if (grp < 2 * NL) {
#pragma unroll
    for (int q = 0; q < P; ++q) L[off + padg<PG>(TPT * q)] = w[0][q];
  }
  lds_barrier();
  const cplx<T>* base = lds + col;
  cplx<T>* S = lds + 2 * NL * BUF + col;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < Y::QN; ++i) {
    if (!mine(i)) continue;
    const int l = row(i), jl = layer(i), s = padg<PG>(l);
    const bool kept = (kept_l(g, l) && kr < g.kmax) || (NL > 1 && c.nomask);
    cplx<T> r = czero<T>();
    if (active && in_col<GEN>(l, ny) && (kept || c.full)) {
      const StagePoint<T> pt = point(i);
      const StageIn<T> one = Y::AHEAD ? in[Y::AHEAD ? i : 0] : stage_load<T>(c, epi, pt);
      // the bottom drag's psih of the calcN input, which the pass that made that input left (k3_body)
      const cplx<T> psin = NL > 1 && c.drag_src != nullptr && jl == NL - 1 && kept ? at(c.psi_in, pt.idx) : czero<T>();
      r = stage_point<T, NL, false, true>(c, epi, pt, one, kept, jl, kv, lwave(g, l), base[(2 * jl) * BUF + s], base[(2 * jl + 1) * BUF + s], psin,
                                          c.noise + (long)jl * (c.fkx + 1) * c.nbl, bad);
    }
    S[jl * BUF + s] = r;
  }
  const unsigned long long badm = __ballot(bad);
  if (badm != 0 && c.nonfinite != nullptr && (int)(threadIdx.x & 63) == __ffsll(badm) - 1) *c.nonfinite = 1;
  if (a.ncols == 0) return;                            // the last stage of a call
  lds_barrier();

  // group 3 jl + f: field f (u, v, q) of layer jl of the next calcN!
  const int jl = grp / 3, field = grp % 3;
  const bool out = active && kr < a.ncols;
  cplx<T> sv[P];
  if (field == 2) {
#pragma unroll
    for (int q = 0; q < P; ++q) sv[q] = S[jl * BUF + off + padg<PG>(TPT * q)];
  } else if constexpr (NL == 1) {
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int l = t + TPT * q;
      const cplx<T> s = S[off + padg<PG>(TPT * q)];
      sv[q] = MODEL == M_TWODNS ? rmul(-inv_k2(kr, l, kv, lwave(g, l)), s) : slqg_psi(a.eb, a.ell2inv, s, kr, l, kv, lwave(g, l));
    }
  } else {
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const T* mm = a.sinv + boff(krl, safe(t + TPT * q), ny) * (NL * NL) + jl * NL;
      cplx<T> acc = czero<T>();
#pragma unroll
      for (int k = 0; k < NL; ++k) acc = rfma(mm[k], S[k * BUF + off + padg<PG>(TPT * q)], acc);
      sv[q] = acc;
    }
    if (field == 0 && jl == NL - 1 && a.psi_out != nullptr && out) {
#pragma unroll
      for (int q = 0; q < P; ++q)
        if (in_col<GEN>(t + TPT * q, ny)) at(a.psi_out, boff32(kr, t + TPT * q, ny)) = sv[q];
    }
  }
  lds_barrier();                                       // the modes are read: the buffers are free
  const T nrm = g.inv_norm;
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const cplx<T> r = field == 2 ? sv[q] : k1_field(field == 0 ? F_U : F_V, sv[q], kv, lwave(g, t + TPT * q));
    w[0][q] = mk(r.re * nrm, -(r.im * nrm));
  }
  y_transform<T, NY, P, false, GEN, X_WAVE>(w, L, t, tw, ny);
  if (out) {
    cplx<T>* o = a.out + (long)(3 * jl + field) * a.fstride;
#pragma unroll
    for (int q = 0; q < P; ++q)
      if (in_col<GEN>(t + TPT * q, ny)) at(o, boff32(kr, t + TPT * q, ny)) = conj(w[0][q]);
  }
}

template <typename T, int NY, int NL, int MODEL, bool GEN>
void ylayers_go(const K3Args<T>& c, const K1Args<T>& a, hipStream_t s) {
  constexpr int P = ylayers_p(NY), CPW = k3_single_column(NY, P) ? 1 : 2;
  const int nblk = CPW == 1 ? column_blocks(c.ncols) : pair_blocks(c.ncols, YL<T, NY, P, NL, CPW, GEN>::G);
  if (c.ncols <= 0) return;
  GF_LAUNCH((ylayers_kernel<T, NY, P, NL, CPW, MODEL, GEN>), dim3(nblk), dim3(64 * 3 * NL), 0, s, c, a);
}
template <typename T, int NY, bool GEN>
void ylayers_l(const K3Args<T>& c, const K1Args<T>& a, hipStream_t s) {
  if (c.model != M_MLQG) {
    if constexpr (GEN) {
      if (c.model == M_TWODNS) ylayers_go<T, NY, 1, M_TWODNS, true>(c, a, s);
      else ylayers_go<T, NY, 1, M_SLQG, true>(c, a, s);
    }
    return;
  }
  switch (c.g.nlayers) {
    case 2: ylayers_go<T, NY, 2, M_MLQG, GEN>(c, a, s); break;
    case 3: ylayers_go<T, NY, 3, M_MLQG, GEN>(c, a, s); break;
    case 4: ylayers_go<T, NY, 4, M_MLQG, GEN>(c, a, s); break;
    case 5: ylayers_go<T, NY, 5, M_MLQG, GEN>(c, a, s); break;
    default: break;
  }
}

}  // namespace gf
