// heom_hilb kernels without matrix cores: the fast path (N = 6..16, diagonal V),
// the general path (N <= 16) and the vector-ALU path of large blocks.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// ---------------------------------------------------------------------------
// heom_hilb, fast path: one ADO per workgroup (N = 6..16), diagonal V
// (heom_hilb.h:96-212 with [V,X]_ij = (v_i - v_j) X_ij, {V,X}_ij = (v_i + v_j) X_ij)
//
// Workgroup b takes the ADO of work unit bmap[b] (its link range in the same
// record), read beside the control block.  H and the diagonals of every V_u
// are staged in LDS once per ADO (no per-link coefficient tables), each link is
// an 8-byte scalar record, its coefficient-table entry and one neighbour-element
// load (the 64-byte LinkFlat records cost 8% more time per stage).
// REAL: H and every V_u real (the commutator and the link coefficients in real
// arithmetic on the real parts; a complex H or V takes REAL = false).
// ---------------------------------------------------------------------------
template <int N>
struct WaveCfg {
  static constexpr int N2 = N * N;
  static constexpr int BS = ((N2 + 63) / 64) * 64;
};

// LDS bytes of the diagonals of every V_u (plus one zero row for direct links)
inline size_t fast_vd_lds(const FormDev& d, bool real, int real_bytes) {
  const size_t rows = static_cast<size_t>(d.n_noise + 1) * d.N;
  return rows * (real ? 1 : 2) * static_cast<size_t>(real_bytes);
}
template <int N, typename R, bool REAL, bool F64, int KP, Epi E>
__global__ void __launch_bounds__(WaveCfg<N>::BS, 1)
    hilb_fast_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  using HT = typename std::conditional<REAL, R, C>::type;
  constexpr int N2 = N * N, BS = WaveCfg<N>::BS;
  __shared__ C s_rho[N2];
  __shared__ HT s_H[N2];
  extern __shared__ __align__(16) unsigned char s_dyn[];
  R* s_vr = reinterpret_cast<R*>(s_dyn);  // real V: v_u,i at u*N + i
  C* s_vc = reinterpret_cast<C*>(s_dyn);  // complex V

  const auto bmp = cst(d.bmap) + blockIdx.x;
  const BlockMap bm{bmp->g, bmp->l0, bmp->l1, 0};
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const int e = threadIdx.x;
  const bool lane_ok = e < N2;
  const int ee = lane_ok ? e : 0;
  const int i = ee / N, j = ee - (ee / N) * N;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const auto lks = cst(d.links);
  const auto cfs = cst(d.coef);

  // idle lanes (e >= N2) read element 0 and store nothing
  const int g = bm.g;
  const long long gi = static_cast<long long>(g) * N2 + ee;
  const int nvd = (d.n_noise + 1) * N, nvd0 = d.n_noise * N;
  const z128 hv = d.H[ee];  // BS >= N2: one element of H per lane
  const z128 vdv = e < nvd0 ? d.Vd[e] : z128{0.0, 0.0};
  const C dterm = conv<R>(d.dterm[ee]);
  const C r = in[gi];
  const int l0 = bm.l0, l1 = bm.l1;
  // the wide-operand stages issue their first four links before the barrier
  // (measured: faster there, slower for stages of at most four operands)
  const int nb0 = KP > 4 ? ((l1 - l0 < 4) ? l1 - l0 : 4) : 0;
  LinkFlat q[4];
  C x[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t < nb0) {
      q[t] = ld_link_coef(lks, cfs, l0 + t);
      x[t] = in[static_cast<long long>(q[t].nbr) * N2 + ee];
    }
  }
  PreT<KP> pv;
  // stages of at most four epilogue operands load them here, ahead of the
  // operator work; the wider stages load them after the links (76 instead of 87
  // VGPRs in FP64: six waves per SIMD instead of five; measured faster there)
  if constexpr (KP <= 4) prefetch<F64, KP>(pv, A, cur, gi, true);
  const C gm = conv<R>(z128{cst(d.gam)[g].re, cst(d.gam)[g].im});
  // LDS: H, the diagonals of V (zero row for direct links last), rho_n
  if (lane_ok) {
    if constexpr (REAL)
      s_H[e] = static_cast<R>(hv.re);
    else
      s_H[e] = conv<R>(hv);
  }
  for (int xx = e; xx < nvd; xx += BS) {
    const z128 v = xx == e ? vdv : (xx < nvd0 ? d.Vd[xx] : z128{0.0, 0.0});
    if (REAL)
      s_vr[xx] = static_cast<R>(v.re);
    else
      s_vc[xx] = conv<R>(v);
  }
  if (lane_ok) s_rho[e] = r;
  __syncthreads();

  C acc{0, 0};
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const C b = s_rho[k * N + j], t = s_rho[i * N + k];
    if constexpr (REAL) {
      const R hik = s_H[i * N + k], hkj = s_H[k * N + j];
      acc.re += hik * b.re;
      acc.im += hik * b.im;
      acc.re -= t.re * hkj;
      acc.im -= t.im * hkj;
    } else {
      cmac(acc, s_H[i * N + k], b);
      cmac(acc, C{-t.re, -t.im}, s_H[k * N + j]);
    }
  }
  C D = times_i(acc);
  cmac(D, gm + dterm, r);
  // link l adds ((v_i - v_j) i*phi + (v_i + v_j) psi + dir) X_nbr, in link order
  auto apply = [&](const LinkFlat& lq, const C& xv) {
    C w;
    if constexpr (REAL) {
      const R vi = s_vr[lq.u * N + i], vj = s_vr[lq.u * N + j];
      const R c0 = vi - vj, a0 = vi + vj;
      w.re = c0 * static_cast<R>(lq.iphi.re) + a0 * static_cast<R>(lq.psi.re) +
             static_cast<R>(lq.dir.re);
      w.im = c0 * static_cast<R>(lq.iphi.im) + a0 * static_cast<R>(lq.psi.im) +
             static_cast<R>(lq.dir.im);
    } else {
      const C vi = s_vc[lq.u * N + i], vj = s_vc[lq.u * N + j];
      w = (vi - vj) * conv<R>(lq.iphi) + (vi + vj) * conv<R>(lq.psi) + conv<R>(lq.dir);
    }
    cmac(D, w, xv);
  };
#pragma unroll
  for (int t = 0; t < 4; ++t)
    if (t < nb0) apply(q[t], x[t]);
  for (int l = l0 + nb0; l < l1; l += 4) {
    const int nb = (l1 - l < 4) ? l1 - l : 4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t < nb) {
        q[t] = ld_link_coef(lks, cfs, l + t);
        x[t] = in[static_cast<long long>(q[t].nbr) * N2 + ee];
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (t < nb) apply(q[t], x[t]);
  }
  if constexpr (KP > 4) prefetch<F64, KP>(pv, A, cur, gi, true);
  double w2 = 0.0;
  if (lane_ok) {
    add_closure(d, gi, D);
    w2 = epilogue<F64, R, KP, E>(pv, A, cur, gi, D, pg.alpha);
  }
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, w2);
}

// ---------------------------------------------------------------------------
// heom_hilb, general path: any V, N <= 16; N <= 8 packs 64/N^2 ADOs per
// wavefront (heom_hilb.h:96-212).  N = 16 in FP32 is held to four waves per SIMD: with
// dense V the compiler otherwise takes 137 registers (924 ADOs, RK4 pass: 32.5 us, 24.4 us
// bounded); other sizes are as fast or faster unbounded.
// ---------------------------------------------------------------------------
template <int N>
struct HilbCfg {
  static constexpr int N2 = N * N;
  static constexpr int BS = N2 <= 64 ? 64 : ((N2 + 63) / 64) * 64;
  static constexpr int APB = BS / N2;  // ADOs per workgroup
};

template <int N, typename R, bool DIAGV, bool F64, int KP, Epi E>
__global__ void __launch_bounds__(HilbCfg<N>::BS, N == 16 && sizeof(R) == 4 ? 4 : 1)
    hilb_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  constexpr int N2 = N * N, APB = HilbCfg<N>::APB, BS = HilbCfg<N>::BS;
  __shared__ C s_rho[APB * N2];
  __shared__ C s_H[N2];
  __shared__ C s_X[DIAGV ? 1 : APB * N2];
  __shared__ C s_Y[DIAGV ? 1 : APB * N2];
  extern __shared__ __align__(16) unsigned char s_dyn[];
  C* s_vd = reinterpret_cast<C*>(s_dyn);

  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const int tid = threadIdx.x;
  const int la = tid / N2;
  const int e = tid - la * N2;
  const int i = e / N, j = e - (e / N) * N;
  const bool lane_ok = la < APB;
  for (int x = tid; x < N2; x += BS) s_H[x] = conv<R>(d.H[x]);
  if (DIAGV) {
    // diagonal of every V_u, then one zero row for direct (off-diagonal gamma) links
    for (int x = tid; x < (d.n_noise + 1) * N; x += BS)
      s_vd[x] = x < d.n_noise * N ? conv<R>(d.Vd[x]) : C{0, 0};
  }
  const C dterm = (DIAGV && lane_ok) ? conv<R>(d.dterm[e]) : C{0, 0};
  const C* in = static_cast<const C*>(pick(A.in, cur));

  double err_acc = 0.0;
  const int n_groups = (d.n_hrchy + APB - 1) / APB;
  for (int g = blockIdx.x; g < n_groups; g += gridDim.x) {
    const int n = g * APB + la;
    const bool ok = lane_ok && n < d.n_hrchy;
    const long long gi = static_cast<long long>(n) * N2 + e;
    const C r = ok ? in[gi] : C{0, 0};
    PreT<KP> pv;
    prefetch<F64, KP>(pv, A, cur, gi, ok);
    const int l0 = ok ? d.link_ptr[n] : 0;
    const int l1 = ok ? d.link_ptr[n + 1] : 0;
    if (lane_ok) s_rho[tid] = r;
    __syncthreads();
    C acc{0, 0};
    if (lane_ok) {
      const C* b = s_rho + la * N2;
#pragma unroll
      for (int k = 0; k < N; ++k) {
        cmac(acc, s_H[i * N + k], b[k * N + j]);
        const C t = b[i * N + k];
        cmac(acc, C{-t.re, -t.im}, s_H[k * N + j]);
      }
    }
    C D = times_i(acc);
    if (ok) cmac(D, conv<R>(d.gam[n]) + dterm, r);
    if (DIAGV) {
      int l = l0;
      for (; l + 2 <= l1; l += 2) {
        const LinkFlat q0 = d.flat[l], q1 = d.flat[l + 1];
        const C x0 = in[static_cast<long long>(q0.nbr) * N2 + e];
        const C x1 = in[static_cast<long long>(q1.nbr) * N2 + e];
        const C vi0 = s_vd[q0.u * N + i], vj0 = s_vd[q0.u * N + j];
        const C vi1 = s_vd[q1.u * N + i], vj1 = s_vd[q1.u * N + j];
        cmac(D, (vi0 - vj0) * conv<R>(q0.iphi) + (vi0 + vj0) * conv<R>(q0.psi) + conv<R>(q0.dir),
             x0);
        cmac(D, (vi1 - vj1) * conv<R>(q1.iphi) + (vi1 + vj1) * conv<R>(q1.psi) + conv<R>(q1.dir),
             x1);
      }
      for (; l < l1; ++l) {
        const LinkFlat q0 = d.flat[l];
        const C x0 = in[static_cast<long long>(q0.nbr) * N2 + e];
        const C vi0 = s_vd[q0.u * N + i], vj0 = s_vd[q0.u * N + j];
        cmac(D, (vi0 - vj0) * conv<R>(q0.iphi) + (vi0 + vj0) * conv<R>(q0.psi) + conv<R>(q0.dir),
             x0);
      }
    } else {
      // dense V: Phi_u, Psi_u per noise, then V_u X + Y V_u (heom_hilb.h:113-208)
      int l = l0;
      for (int u = 0; u < d.n_noise; ++u) {
        C phi{0, 0}, psi{0, 0};
        while (l < l1) {
          const Link lk = d.links[l];
          const Coef c = d.coef[lk.cid];
          if (c.u != u) break;
          const C x = in[static_cast<long long>(lk.nbr) * N2 + e];
          cmac(phi, conv<R>(c.phi), x);
          cmac(psi, conv<R>(c.psi), x);
          ++l;
        }
        const z128* V = d.V + static_cast<long long>(u) * N2;
        C cc{0, 0};
        if (lane_ok) {
          const C* b = s_rho + la * N2;
#pragma unroll
          for (int k = 0; k < N; ++k) {
            cmac(cc, conv<R>(V[i * N + k]), b[k * N + j]);
            const C t = b[i * N + k];
            cmac(cc, C{-t.re, -t.im}, conv<R>(V[k * N + j]));
          }
        }
        const C sd = conv<R>(d.sdelta[u]);
        const C dcc = sd * cc;
        const C iphi = times_i(phi);
        // i[V,Phi] + {V,Psi} + delta[V,[V,rho]] = V X + Y V
        const C X = iphi + psi + dcc;
        const C Y = psi - iphi - dcc;
        if (lane_ok) {
          s_X[tid] = X;
          s_Y[tid] = Y;
        }
        __syncthreads();
        if (lane_ok) {
          const C* bx = s_X + la * N2;
          const C* by = s_Y + la * N2;
#pragma unroll
          for (int k = 0; k < N; ++k) {
            cmac(D, conv<R>(V[i * N + k]), bx[k * N + j]);
            cmac(D, by[i * N + k], conv<R>(V[k * N + j]));
          }
        }
        __syncthreads();
      }
      for (; l < l1; ++l) {
        const Link lk = d.links[l];
        const Coef c = d.coef[lk.cid];
        cmac(D, conv<R>(c.dir), in[static_cast<long long>(lk.nbr) * N2 + e]);
      }
    }
    if (ok) {
      add_closure(d, gi, D);
      err_acc += epilogue<F64, R, KP, E>(pv, A, cur, gi, D, pg.alpha);
    }
    __syncthreads();
  }
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, err_acc);
}

// ---------------------------------------------------------------------------
// heom_hilb, large N (N > 16), diagonal V: one ADO per workgroup of 256 lanes,
// each lane owns a 4x4 tile of elements.  The block sits in LDS (and H too
// when both fit in 64 KB); the commutator is a register-tiled complex matrix
// product, the neighbour terms and the stage epilogue run per owned element.
// ---------------------------------------------------------------------------
constexpr int kBigBS = 256;
constexpr int kBigTile = 4;

template <typename R, bool HLDS, bool F64, int KP, Epi E>
__global__ void __launch_bounds__(kBigBS) hilb_big_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  extern __shared__ __align__(16) unsigned char s_dyn[];
  const int N = d.N, N2 = d.N2;
  C* s_rho = reinterpret_cast<C*>(s_dyn);
  C* s_H = s_rho + N2;
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const auto link_ptr = cst(d.link_ptr);
  const auto flat = cst(d.flat);
  const auto gam = cst(d.gam);
  const int nt = (N + kBigTile - 1) / kBigTile;  // tiles per row
  if (HLDS)
    for (int x = threadIdx.x; x < N2; x += kBigBS) s_H[x] = conv<R>(d.H[x]);
  double err_acc = 0.0;
  for (int g = blockIdx.x; g < d.n_hrchy; g += gridDim.x) {
    const long long base = static_cast<long long>(g) * N2;
    for (int x = threadIdx.x; x < N2; x += kBigBS) s_rho[x] = in[base + x];
    __syncthreads();
    const int l0 = link_ptr[g], l1 = link_ptr[g + 1];
    const C gm = conv<R>(z128{gam[g].re, gam[g].im});
    for (int t = threadIdx.x; t < nt * nt; t += kBigBS) {
      const int r0 = (t / nt) * kBigTile, c0 = (t % nt) * kBigTile;
      C acc[kBigTile][kBigTile];
#pragma unroll
      for (int a = 0; a < kBigTile; ++a)
#pragma unroll
        for (int b = 0; b < kBigTile; ++b) acc[a][b] = C{0, 0};
      for (int k = 0; k < N; ++k) {
        C hr[kBigTile], rr[kBigTile], rc[kBigTile], hc[kBigTile];
#pragma unroll
        for (int a = 0; a < kBigTile; ++a) {
          const int i = r0 + a < N ? r0 + a : N - 1;
          const int j = c0 + a < N ? c0 + a : N - 1;
          hr[a] = HLDS ? s_H[i * N + k] : conv<R>(d.H[i * N + k]);
          rc[a] = s_rho[i * N + k];
          rr[a] = s_rho[k * N + j];
          hc[a] = HLDS ? s_H[k * N + j] : conv<R>(d.H[k * N + j]);
        }
#pragma unroll
        for (int a = 0; a < kBigTile; ++a)
#pragma unroll
          for (int b = 0; b < kBigTile; ++b) {
            cmac(acc[a][b], hr[a], rr[b]);
            cmac(acc[a][b], C{-rc[a].re, -rc[a].im}, hc[b]);
          }
      }
#pragma unroll
      for (int a = 0; a < kBigTile; ++a)
#pragma unroll
        for (int b = 0; b < kBigTile; ++b) {
          const int i = r0 + a, j = c0 + b;
          if (i >= N || j >= N) continue;
          const int e = i * N + j;
          const C r = s_rho[e];
          C D = times_i(acc[a][b]);
          cmac(D, gm + conv<R>(d.dterm[e]), r);
          for (int l = l0; l < l1; ++l) {
            const LinkFlat q = ld_flat(flat + l);
            const C x = in[static_cast<long long>(q.nbr) * N2 + e];
            const long long tb = static_cast<long long>(q.u) * N2 + e;
            C cf;
            if (d.real_v) {
              const z128 p = d.cmac_tab[tb];
              cf.re = static_cast<R>(p.re) * static_cast<R>(q.iphi.re) +
                      static_cast<R>(p.im) * static_cast<R>(q.psi.re) + static_cast<R>(q.dir.re);
              cf.im = static_cast<R>(p.re) * static_cast<R>(q.iphi.im) +
                      static_cast<R>(p.im) * static_cast<R>(q.psi.im) + static_cast<R>(q.dir.im);
            } else {
              cf = conv<R>(d.cmac_tab[2 * tb]) * conv<R>(q.iphi) +
                   conv<R>(d.cmac_tab[2 * tb + 1]) * conv<R>(q.psi) + conv<R>(q.dir);
            }
            cmac(D, cf, x);
          }
          PreT<KP> pv;
          prefetch<F64, KP>(pv, A, cur, base + e, true);
          add_closure(d, base + e, D);
          err_acc += epilogue<F64, R, KP, E>(pv, A, cur, base + e, D, pg.alpha);
        }
    }
    __syncthreads();
  }
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, err_acc);
}

template <int N, typename R, bool F64>
int launch_hilb_n(const FormDev& d, const StageArgs& A, hipStream_t st) {
  if (N >= 4 && d.slinks != nullptr) return launch_hilb_split<R, F64>(d, A, st);
  if constexpr (N >= 6) {
    const bool real = d.real_v && d.real_h;
    const size_t lds = fast_vd_lds(d, real, sizeof(R));
    if (d.diag_v && d.bmap != nullptr && d.n_hrchy <= kMaxGrid && lds <= 32 * 1024) {
      const int grid = d.n_hrchy;
      // four prefetched operands cover every stage but Dormand-Prince's fifth and sixth
      const auto run = [&](auto real_, auto kp, auto epi) {
        hipLaunchKernelGGL(
            (hilb_fast_kernel<N, R, decltype(real_)::value, F64, decltype(kp)::value,
                              decltype(epi)::value>),
            dim3(grid), dim3(WaveCfg<N>::BS), lds, st, d, A);
      };
      if (real)
        with_epilogue<4, 6>(A, [&](auto kp, auto epi) { run(std::true_type{}, kp, epi); });
      else
        with_epilogue<4, kMaxPre>(A, [&](auto kp, auto epi) { run(std::false_type{}, kp, epi); });
      return grid;
    }
  }
  constexpr int APB = HilbCfg<N>::APB, BS = HilbCfg<N>::BS;
  const int grid = cap_grid((d.n_hrchy + APB - 1) / APB);
  const size_t lds = d.diag_v ? sizeof(cx<R>) * (d.n_noise + 1) * N : 0;
  if (lds > 48 * 1024)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "heom_hilb: too many noises for the LDS tables"};
  with_epilogue<4, kMaxPre>(A, [&](auto kp, auto epi) {
    constexpr int KP = decltype(kp)::value;
    constexpr Epi E = decltype(epi)::value;
    if (d.diag_v)
      hipLaunchKernelGGL((hilb_kernel<N, R, true, F64, KP, E>), dim3(grid), dim3(BS), lds, st, d,
                         A);
    else
      hipLaunchKernelGGL((hilb_kernel<N, R, false, F64, KP, E>), dim3(grid), dim3(BS), 0, st, d,
                         A);
  });
  return grid;
}
template <typename R, bool F64>
int launch_hilb_big(const FormDev& d, const StageArgs& A, hipStream_t st) {
  if (d.mfma == 3)  // 16 < N <= 64, dense V
    return launch_hilb_mfma_dense<R, F64>(d, A, st);
  if (d.mfma) return launch_hilb_mfma<R, F64>(d, A, st);  // 16 < N <= 64, diagonal V
  if (!d.diag_v)
    throw HeomError{HEOM_ERR_UNSUPPORTED,
                    "heom_hilb: n_level > 16 is provided for diagonal coupling operators V"};
  const size_t one = sizeof(cx<R>) * static_cast<size_t>(d.N2);
  const int grid = cap_grid(d.n_hrchy);
  if (one > 64 * 1024)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "heom_hilb: one ADO block exceeds 64 KB of LDS"};
  with_epilogue<4, kMaxPre>(A, [&](auto kp, auto epi) {
    constexpr int KP = decltype(kp)::value;
    constexpr Epi E = decltype(epi)::value;
    if (2 * one <= 64 * 1024)
      hipLaunchKernelGGL((hilb_big_kernel<R, true, F64, KP, E>), dim3(grid), dim3(kBigBS),
                         2 * one, st, d, A);
    else
      hipLaunchKernelGGL((hilb_big_kernel<R, false, F64, KP, E>), dim3(grid), dim3(kBigBS), one,
                         st, d, A);
  });
  return grid;
}

}  // namespace

template <typename R, bool F64>
int launch_hilb(const FormDev& d, const StageArgs& A, hipStream_t st) {
  switch (d.N) {
#define HAMD_CASE(n) \
  case n:            \
    return launch_hilb_n<n, R, F64>(d, A, st);
    HAMD_CASE(1) HAMD_CASE(2) HAMD_CASE(3) HAMD_CASE(4) HAMD_CASE(5) HAMD_CASE(6) HAMD_CASE(7)
    HAMD_CASE(8) HAMD_CASE(9) HAMD_CASE(10) HAMD_CASE(11) HAMD_CASE(12) HAMD_CASE(13)
    HAMD_CASE(14) HAMD_CASE(15) HAMD_CASE(16)
#undef HAMD_CASE
    default:
      return launch_hilb_big<R, F64>(d, A, st);
  }
}

HAMD_FORM_INSTANCES(launch_hilb)

}  // namespace hamd
