// heom_hilb with diagonal V, 4 <= N <= 16: the links of an ADO with many are
// shared between the groups of lanes of its workgroup.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// ---------------------------------------------------------------------------
// A workgroup is G groups of lanes, one lane per element, and takes one work
// unit: G ADOs with few links, a group each, or one ADO with many, whose links
// and commutator the groups share (their sums meet in LDS, group 0 adds them in
// order).  The ADOs above the last tier have a link per mode (22 on the 7-site
// chain with 21 modes, where the last tier has at most its depth), and a group
// that takes them four at a time (hilb_fast_kernel) makes a trip to the link
// records and one to the neighbours for each four: on a small hierarchy that
// chain is the stage.  Here a group's links are one round, up to kSplitRound of
// them, and its records lie in slots of fixed length, so their address is known
// without the work unit.  Lanes of a group are whole wavefronts from N = 6 on
// (scalar records).  Bound: latency (launch, record, neighbour, store).  RK4 stage
// with its launch: 253 ADOs of 7x7 9.8 -> 5.6 us, 495 of 4x4 7.0 -> 5.2 us; where it
// is used: Qme::build_split_units.
// ---------------------------------------------------------------------------
constexpr int kSplitRound = 6;  // links per group and round

template <int N>
struct SplitCfg {
  static constexpr int N2 = N * N, G = split_groups(N);
  static constexpr int lanes = N == 4 ? 16 : N == 5 ? 32 : ((N2 + 63) / 64) * 64;
  static constexpr int BS = lanes * G;
};

template <int N, typename R, bool REAL, bool F64, int KP, Epi E>
__global__ void __launch_bounds__(SplitCfg<N>::BS)
    hilb_split_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  using HT = typename std::conditional<REAL, R, C>::type;
  constexpr int N2 = N * N, G = SplitCfg<N>::G, L = SplitCfg<N>::lanes, BS = SplitCfg<N>::BS;
  __shared__ C s_rho[G * N2];
  __shared__ C s_part[(G - 1) * N2];
  __shared__ HT s_H[N2];
  extern __shared__ __align__(16) unsigned char s_dyn[];
  HT* s_v = reinterpret_cast<HT*>(s_dyn);  // v_u,i at u*N + i, then a zero row

  const int tid = threadIdx.x;
  const int q = L >= 64 ? __builtin_amdgcn_readfirstlane(tid / L) : tid / L;
  const int e = tid - q * L;
  const int unit = blockIdx.x * G + q;
  // the group's ADO (-1: none); a shared one is marked in the workgroup's first record
  const bool heavy = cst(d.sunits)[blockIdx.x * G].shared != 0;
  int g;
  if constexpr (L >= 64)
    g = cst(d.sunits)[unit].g;
  else
    g = d.sunits[unit].g;
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const bool ok = e < N2 && g >= 0;
  const int ee = e < N2 ? e : 0;
  const int i = ee / N, j = ee - (ee / N) * N;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const Link* slots = d.slinks + static_cast<long long>(unit) * d.slink_n;
  const long long gi = static_cast<long long>(g < 0 ? 0 : g) * N2 + ee;

  // the links of a round: records, then neighbours
  int nbr[kSplitRound], cid[kSplitRound];
  C x[kSplitRound];
  auto load = [&](int first) {
#pragma unroll
    for (int t = 0; t < kSplitRound; ++t) {
      nbr[t] = -1;
      if (first + t < d.slink_n) {
        if constexpr (L >= 64) {
          nbr[t] = cst(slots)[first + t].nbr;
          cid[t] = cst(slots)[first + t].cid;
        } else {
          const Link k = slots[first + t];
          nbr[t] = k.nbr;
          cid[t] = k.cid;
        }
      }
    }
#pragma unroll
    for (int t = 0; t < kSplitRound; ++t)
      if (nbr[t] >= 0) x[t] = in[static_cast<long long>(nbr[t]) * N2 + ee];
  };
  load(0);
  // one group owns the element: its own, or group 0 of a shared ADO
  const bool own = ok && (!heavy || q == 0);
  C r{0, 0}, gd{0, 0};
  PreT<KP> pv;
  if (own) {
    r = in[gi];
    if constexpr (KP <= 4) prefetch<F64, KP>(pv, A, cur, gi, true);
    gd = conv<R>(d.gam[g]) + conv<R>(d.dterm[ee]);
  }
  const int nvd = (d.n_noise + 1) * N, nvd0 = d.n_noise * N;
  for (int t = tid; t < N2 + nvd; t += BS) {
    const z128 v = t < N2 ? d.H[t] : (t - N2 < nvd0 ? d.Vd[t - N2] : z128{0.0, 0.0});
    HT w;
    if constexpr (REAL)
      w = static_cast<R>(v.re);
    else
      w = conv<R>(v);
    if (t < N2)
      s_H[t] = w;
    else
      s_v[t - N2] = w;
  }
  C* s_r = s_rho + (heavy ? 0 : q * N2);
  if (own) s_r[e] = r;
  __syncthreads();

  // link l adds ((v_i - v_j) i*phi + (v_i + v_j) psi + dir) X_nbr
  C D{0, 0};
  auto apply = [&](int c, const C& xv) {
    z128 phi, psi, dir;
    int u;
    if constexpr (L >= 64) {
      const auto cf = cst(d.coef) + c;
      phi = z128{cf->phi.re, cf->phi.im};
      psi = z128{cf->psi.re, cf->psi.im};
      dir = z128{cf->dir.re, cf->dir.im};
      u = cf->u;
    } else {
      const Coef cf = d.coef[c];
      phi = cf.phi;
      psi = cf.psi;
      dir = cf.dir;
      u = cf.u;
    }
    const z128 iphi{-phi.im, phi.re};
    C w;
    if constexpr (REAL) {
      const R vi = s_v[u * N + i], vj = s_v[u * N + j];
      const R c0 = vi - vj, a0 = vi + vj;
      w.re = c0 * static_cast<R>(iphi.re) + a0 * static_cast<R>(psi.re) + static_cast<R>(dir.re);
      w.im = c0 * static_cast<R>(iphi.im) + a0 * static_cast<R>(psi.im) + static_cast<R>(dir.im);
    } else {
      const C vi = s_v[u * N + i], vj = s_v[u * N + j];
      w = (vi - vj) * conv<R>(iphi) + (vi + vj) * conv<R>(psi) + conv<R>(dir);
    }
    cmac(D, w, xv);
  };
  // products k = k0, k0 + kd, ... of H rho - rho H
  C acc{0, 0};
  auto product = [&](int k) {
    const C b = s_r[k * N + j], t = s_r[i * N + k];
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
  };
  if (heavy) {
    for (int k = q; k < N; k += G) product(k);
  } else {
#pragma unroll
    for (int k = 0; k < N; ++k) product(k);
  }
  for (int first = 0;;) {
#pragma unroll
    for (int t = 0; t < kSplitRound; ++t)
      if (nbr[t] >= 0) apply(cid[t], x[t]);
    first += kSplitRound;
    if (first >= d.slink_n) break;
    load(first);
  }
  D = D + times_i(acc);
  if constexpr (KP > 4)
    if (own) prefetch<F64, KP>(pv, A, cur, gi, true);
  if (heavy) {
    if (q > 0 && e < N2) s_part[(q - 1) * N2 + e] = D;
    __syncthreads();
    if (own) {
#pragma unroll
      for (int p = 0; p < G - 1; ++p) D = D + s_part[p * N2 + e];
    }
  }
  double w2 = 0.0;
  if (own) {
    cmac(D, gd, r);
    add_closure(d, gi, D);
    w2 = epilogue<F64, R, KP, E>(pv, A, cur, gi, D, pg.alpha);
  }
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, w2);
}

template <int N, typename R, bool F64>
int launch_split_n(const FormDev& d, const StageArgs& A, hipStream_t st) {
  const bool real = d.real_v && d.real_h;
  const size_t lds = split_vd_lds(d.n_noise, N, real, sizeof(R));
  const dim3 grid(d.n_sunits), block(SplitCfg<N>::BS);
  with_epilogue<4, 6>(A, [&](auto kp, auto epi) {
    constexpr Epi E = decltype(epi)::value;
    if (real)
      hipLaunchKernelGGL((hilb_split_kernel<N, R, true, F64, decltype(kp)::value, E>), grid,
                         block, lds, st, d, A);
    else
      hipLaunchKernelGGL((hilb_split_kernel<N, R, false, F64, 6, E>), grid, block, lds, st, d, A);
  });
  return d.n_sunits;
}

}  // namespace

template <typename R, bool F64>
int launch_hilb_split(const FormDev& d, const StageArgs& A, hipStream_t st) {
  switch (d.N) {
#define HAMD_CASE(n) \
  case n:            \
    return launch_split_n<n, R, F64>(d, A, st);
    HAMD_CASE(4) HAMD_CASE(5) HAMD_CASE(6) HAMD_CASE(7) HAMD_CASE(8) HAMD_CASE(9) HAMD_CASE(10)
    HAMD_CASE(11) HAMD_CASE(12) HAMD_CASE(13) HAMD_CASE(14) HAMD_CASE(15) HAMD_CASE(16)
#undef HAMD_CASE
    default:
      throw HeomError{HEOM_ERR_STATE, "hilb_split: n_level outside 4..16"};
  }
}

HAMD_FORM_INSTANCES(launch_hilb_split)

}  // namespace hamd
