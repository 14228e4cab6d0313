// The fused y pass of consecutive calcN! evaluations: K3 of one stage and K1 of the next.
//
// Both work on whole kr columns: K3 transforms a column's fluxes forward along y and steps its
// modes, K1 reads those modes back, forms u, v and q and transforms them inversely.  Inside a
// run of stages one kernel does both, so a stage is two launches (x pass, y pass) instead of
// three, the new state is not read back, and the intermediate states of ETDRK4 that only the
// next K1 reads (stages 2 and 3) are not written at all.  The first stage of a call starts with K1;
// the last one's launch leaves the fields out (K1's ncols = 0).  Every expression is the one K3 and K1
// evaluate (stage_point, k1_field), so the results are theirs bit for bit.
//
// NG = 3: three thread groups per column (or column pairs).  Groups 0 and 1 transform the two fluxes
// side by side, the modes of the column are stepped by all three, and each transforms one of u, v, q:
// two transforms in a row where K3 and K1 run five.  Where a group is one wave the transforms need no
// barriers (X_WAVE).  This serves the grids whose y passes wait on latency.
// NG = 1: one group does all five, the state in registers in between: for grids that fill the GPU with
// one group per column already.
//
// FP64 per launch, K3 + K1 -> fused: 64^2 5.8 + 3.4 -> 5.1 us, 128^2 6.6 + 3.6 -> 6.0, 512^2 10.3 + 6.1 -> 12.3,
// 2048^2 (ETDRK4) 26.8 + 21.7 -> 39.6, where it moves 15% less than the two did.
#include "gf_kernels_impl.hpp"

namespace gf {

template <int N, int P, int NG, int CPW> struct YS {
  static constexpr int TPT = N / P;
  static constexpr int G = CPW == 2 ? GY<N, P>::G : 1;
  static constexpr int GT = CPW * G * TPT;             // threads per group, whole waves
  static constexpr int X = GT == 64 ? X_WAVE : X_LDS;
  static constexpr int QN = (P + NG - 1) / NG;         // modes a thread steps
  // single 4096-point columns of 512 threads: two of them fit a CU's LDS, so 4 waves per SIMD are
  // wanted (128 VGPRs, some spilled: 4096^2 RK4 stages 248 -> 212 us)
  static constexpr bool TIGHT = NG == 1 && CPW == 1 && TPT == 512;
};
// Which halves of the fused pass a launch runs: K1 alone (the first stage of a run), both, K3 alone (the
// last).
enum YMode { Y_FIELDS = 0, Y_BOTH = 1, Y_STAGE = 2 };

// LDS of one workgroup, in complex slots (beside the twiddle table).
template <typename T, int N, int P, int NG, int CPW> struct YLds {
  static constexpr int BUF = CPW == 2 ? YS<N, P, NG, CPW>::G * PairLds<T, N>::value : LdsN<N>::value;
  static constexpr int value = NG * BUF;
};

template <typename T, int NY, int P, int NG, int CPW, int MODEL, int EPI, bool AHEAD>
__device__ __forceinline__ void ystage_body(const K3Args<T>& c, const K1Args<T>& a, int blk, int mode, cplx<T>* __restrict__ lds,
                                            cplx<T>* __restrict__ tw) {
  using Y = YS<NY, P, NG, CPW>;
  constexpr int TPT = Y::TPT, G = Y::G, GT = Y::GT, X = Y::X, PG = XPad<T>::G, BUF = YLds<T, NY, P, NG, CPW>::BUF;
  constexpr bool FR = NG == 1 && sizeof(T) == 8 && NY >= 2048;
  constexpr bool TIGHT = Y::TIGHT;
  constexpr int CP = MODEL == M_TWODNS ? 0 : 1;       // real or complex coefficient tables
  const Geo<T>& g = c.g;
  const int grp = NG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / GT);
  const int tid = (int)threadIdx.x % GT;
  int t, kr, col;
  if constexpr (CPW == 2) {
    const YMap<TPT> m(tid);
    t = m.t;
    kr = 2 * (G == 1 ? pair_of_block(blk) : blk * G + m.slot) + m.c;
    col = (int)(col_buffer<T, NY>(lds, m.slot, m.c) - lds);
  } else {
    t = tid;
    kr = single_column(blk);
    col = 0;
  }
  cplx<T>* L = lds + grp * BUF + col;
  const T kv = krwave(g, kr);
  cplx<T> w[1][P], sv[P];
  if (mode == Y_FIELDS) {
    // the state itself, masked
    load_twiddles<T, NY, P>(tw, c.tw);
    const bool in = kr < a.ncols && kr < g.kmax;
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int l = t + TPT * q;
      const cplx<T> v = at(a.sol, boff32(in ? kr : 0, l, NY));
      sv[q] = in && kept_l(g, l) ? v : czero<T>();
    }
    lds_barrier();
  } else {
  const bool active = kr < c.ncols && kr < g.nkr;
  const int epi = EPI >= 0 ? EPI : c.epi;

  // the fluxes of this column: group 0 (u q)^, group 1 (v q)^
  cplx<T> w1[1][NG == 1 ? P : 1];
  const int krl = active ? kr : 0;
  {
    const cplx<T>* f = c.in + (long)(grp == 1 ? c.fstride : 0);
#pragma unroll
    for (int q = 0; q < P; ++q) w[0][q] = at(f, boff32(krl, t + TPT * q, NY));
    if constexpr (NG == 1) {
#pragma unroll
      for (int q = 0; q < P; ++q) w1[0][q] = at(c.in + c.fstride, boff32(krl, t + TPT * q, NY));
    }
  }
  load_twiddles<T, NY, P>(tw, c.tw);
  // what this thread's modes need from memory, under way during the transforms (NG = 3: two or three
  // modes per thread; with one group the registers do not hold them)
  auto row = [&](int i) { return t + TPT * (NG == 1 ? i : grp + NG * i); };
  auto mine = [&](int i) { return NG == 1 || grp + NG * i < P; };
  StageIn<T> in[AHEAD ? Y::QN : 1];
  if constexpr (AHEAD) {
#pragma unroll
    for (int i = 0; i < Y::QN; ++i)
      in[i] = stage_load<T, CP>(c, epi, StagePoint<T>(c, krl, mine(i) ? row(i) : t, NY, 0u));
  }
  // ring forcing: this thread's terms, read back by it in the stage (k3_body)
  if (c.sqrt_spec != nullptr && active && kr <= c.fkx) {
    const int64_t fstep = c.fstep_dev != nullptr ? c.fstep_dev[0] : c.fstep;
    for (int i = 0; i < Y::QN; ++i) {
      const int l = row(i);
      if (mine(i) && (l <= c.fky || l >= NY - c.fky)) {
        const T sp = at(c.sqrt_spec, boff32(kr, l, NY));
        if (sp != (T)0) {
          const cplx<T> xi = complex_normal<T>(c.seed, fstep, (uint32_t)(l * g.nkr + kr), (uint32_t)c.instance);
          c.noise[kr * c.nbl + ring_box_row(l, NY, c.fky, c.nbl)] = mk((xi.re * sp) / c.sqrt_dt, (xi.im * sp) / c.sqrt_dt);
        }
      }
    }
  }
  lds_barrier();                                       // the twiddles
  fft_forward<T, NY, P, 1, FR, X>(w, L, t, tw);
  if constexpr (NG == 1) fft_forward<T, NY, P, 1, FR, X>(w1, L, t, tw);

  bool bad = false;
  if constexpr (NG == 1) {
    // A wait for reads issued after a store waits for the store too (both count in vmcnt), and row by row
    // that chained the P stores' latencies. So each mode's reads are issued before the mode before it stores
    // (PIPE), and the last stage of a step, whose reads would take too many registers for that, stores its new
    // state after the loop (LATE). 2048^2 FP64: ETDRK4 stages 1 and 4 45 and 47 -> 40 and 42 us.
    constexpr bool LATE = EPI == E_ETD4 || EPI == E_RK4 || EPI == E_FE, PIPE = !LATE && !TIGHT;
    // (a row that is not stepped reads the column's first one)
    auto stepped = [&](int l) { return (kept_l(g, l) && kr < g.kmax) || c.full; };
    auto read = [&](int q) {
      const int l = t + TPT * q;
      return stage_load<T, CP>(c, epi, StagePoint<T>(c, krl, stepped(l) ? l : 0, NY, 0u));
    };
    StageIn<T> next;
    if constexpr (PIPE) next = read(0);
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int l = t + TPT * q;
      const bool kept = kept_l(g, l) && kr < g.kmax;
      const StageIn<T> one = PIPE ? next : read(q);
      if (PIPE && q + 1 < P) next = read(q + 1);
      sv[q] = czero<T>();
      if (active && stepped(l))
        sv[q] = stage_point<T, 1, false, true, CP, LATE>(c, epi, StagePoint<T>(c, kr, l, NY, 0u), one, kept, 0, kv, lwave(g, l), w[0][q], w1[0][q],
                                                         czero<T>(), c.noise, bad);
      if constexpr (P >= 8) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LATE) {
      cplx<T>* o = EPI == E_ETD4 && c.sol_out != nullptr ? c.sol_out : c.sol;
#pragma unroll
      for (int q = 0; q < P; ++q) {
        const int l = t + TPT * q;
        if (active && stepped(l)) at(o, boff32(kr, l, NY)) = sv[q];
        if (!(kept_l(g, l) && kr < g.kmax)) sv[q] = czero<T>();
      }
    }
  } else {
    // the transformed fluxes cross groups in buffers 0 and 1, the new modes come back in buffer 2
    const int off = padg<PG>(t);
    if (grp < 2) {
#pragma unroll
      for (int q = 0; q < P; ++q) L[off + padg<PG>(TPT * q)] = w[0][q];
    }
    lds_barrier();
    const cplx<T>* A = lds + col;
    const cplx<T>* B = lds + BUF + col;
    cplx<T>* S = lds + 2 * BUF + col;
#pragma unroll
    for (int i = 0; i < Y::QN; ++i) {
      if (!mine(i)) continue;
      const int l = row(i), s = padg<PG>(l);
      const bool kept = kept_l(g, l) && kr < g.kmax;
      cplx<T> r = czero<T>();
      if (active && (kept || c.full)) {
        const StagePoint<T> pt(c, kr, l, NY, 0u);
        const StageIn<T> one = AHEAD ? in[AHEAD ? i : 0] : stage_load<T, CP>(c, epi, pt);
        r = stage_point<T, 1, false, true, CP>(c, epi, pt, one, kept, 0, kv, lwave(g, l), A[s], B[s], czero<T>(), c.noise, bad);
      }
      S[s] = r;
    }
    lds_barrier();
#pragma unroll
    for (int q = 0; q < P; ++q) sv[q] = S[off + padg<PG>(TPT * q)];
    lds_barrier();                                     // buffer 2 is free
  }
  const unsigned long long badm = __ballot(bad);
  if (badm != 0 && c.nonfinite != nullptr && (int)(threadIdx.x & 63) == __ffsll(badm) - 1) *c.nonfinite = 1;

  if (mode == Y_STAGE) return;
  }

  // the next calcN!'s fields of the kept columns
  const bool out = kr < a.ncols && kr < g.nkr;
  if (CPW == 1 && kr >= a.ncols) return;               // (a single column is its whole workgroup's)
  cplx<T> ps[P];
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int l = t + TPT * q;
    ps[q] = MODEL == M_TWODNS ? rmul(-inv_k2(kr, l, kv, lwave(g, l)), sv[q]) : slqg_psi(a.eb, a.ell2inv, sv[q], kr, l, kv, lwave(g, l));
  }
  const T nrm = g.inv_norm;
#pragma unroll
  for (int f = 0; f < (NG == 1 ? 3 : 1); ++f) {
    // u, v, q (Fields<MODEL, FS_CALCN>); q first where registers are short: after it only psi is held
    const int field = NG > 1 ? grp : (TIGHT ? 2 - f : f);
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const cplx<T> r = field == 2 ? sv[q] : k1_field(field == 0 ? F_U : F_V, ps[q], kv, lwave(g, t + TPT * q));
      w[0][q] = mk(r.re * nrm, -(r.im * nrm));
    }
    fft_forward<T, NY, P, 1, FR, X>(w, L, t, tw);
    if (out) {
      cplx<T>* o = a.out + (long)field * a.fstride;
#pragma unroll
      for (int q = 0; q < P; ++q) at(o, boff32(kr, t + TPT * q, NY)) = conj(w[0][q]);
    }
  }
}

template <typename T, int NY, int P, int NG, int CPW, int MODEL, int EPI>
__global__ __launch_bounds__((NG * YS<NY, P, NG, CPW>::GT)) __attribute__((amdgpu_waves_per_eu((YS<NY, P, NG, CPW>::TIGHT ? 4 : 2))))
void ystage_kernel(const K3Args<T> c, const K1Args<T> a) {
  __shared__ cplx<T> lds[YLds<T, NY, P, NG, CPW>::value];
  __shared__ cplx<T> tw[TwPlan<NY, P>::size()];
  ystage_body<T, NY, P, NG, CPW, MODEL, EPI, (NG > 1)>(c, a, blockIdx.x, a.ncols == 0 ? Y_STAGE : Y_BOTH, lds, tw);
}

template <typename T, int N, int P, int NG, int CPW, int MODEL>
void ystage_go(const K3Args<T>& c, const K1Args<T>& a, hipStream_t s) {
  using Y = YS<N, P, NG, CPW>;
  const int nblk = CPW == 1 ? column_blocks(c.ncols) : pair_blocks(c.ncols, Y::G);
  if (c.ncols <= 0) return;
  const dim3 grid(nblk), blk(NG * Y::GT);
  if constexpr (NG == 1 && N >= 2048) {
    // one kernel per stage: its registers set the occupancy
    switch (c.epi) {
      case E_FE: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_FE>), grid, blk, 0, s, c, a); return;
      case E_AB3: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_AB3>), grid, blk, 0, s, c, a); return;
      case E_RK1: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_RK1>), grid, blk, 0, s, c, a); return;
      case E_RK2: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_RK2>), grid, blk, 0, s, c, a); return;
      case E_RK3: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_RK3>), grid, blk, 0, s, c, a); return;
      case E_RK4: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_RK4>), grid, blk, 0, s, c, a); return;
      case E_ETD1: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_ETD1>), grid, blk, 0, s, c, a); return;
      case E_ETD2: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_ETD2>), grid, blk, 0, s, c, a); return;
      case E_ETD3: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_ETD3>), grid, blk, 0, s, c, a); return;
      case E_ETD4: GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, E_ETD4>), grid, blk, 0, s, c, a); return;
      default: return;
    }
  } else {
    GF_LAUNCH((ystage_kernel<T, N, P, NG, CPW, MODEL, -1>), grid, blk, 0, s, c, a);
  }
}
template <typename T, int N, int P, int NG>
void ystage_p(const K3Args<T>& c, const K1Args<T>& a, hipStream_t s) {
  const bool twodns = c.model == M_TWODNS;
  if constexpr (ystage_built(N, P, NG, 1)) {
    if (c.csplit) {
      if (twodns) ystage_go<T, N, P, NG, 1, M_TWODNS>(c, a, s);
      else ystage_go<T, N, P, NG, 1, M_SLQG>(c, a, s);
      return;
    }
  }
  if constexpr (ystage_built(N, P, NG, 2)) {
    if (twodns) ystage_go<T, N, P, NG, 2, M_TWODNS>(c, a, s);
    else ystage_go<T, N, P, NG, 2, M_SLQG>(c, a, s);
  }
}
template <typename T, int N, int NG>
void ystage_n(const K3Args<T>& c, const K1Args<T>& a, hipStream_t s) {
  switch (c.p ? c.p : sched_default(N)) {
    case 4: ystage_p<T, N, 4, NG>(c, a, s); break;
    case 8: ystage_p<T, N, 8, NG>(c, a, s); break;
    case 16: ystage_p<T, N, 16, NG>(c, a, s); break;
    default: break;
  }
}

}  // namespace gf
