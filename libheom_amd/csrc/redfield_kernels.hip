// The Redfield QMEs, Hilbert and Liouville form.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// ---------------------------------------------------------------------------
// Redfield QMEs (redfield_hilb.h:66-89, redfield_liou.h:91-102):
//   D = i[H, rho] + sum_u [V_u, T_u],  T_u = Lambda_u rho - rho Lambda_u^+
// ---------------------------------------------------------------------------
// One workgroup holds the whole problem (n_level <= 16 and every table within
// 60 KB of LDS), one lane per element.  Every table is staged into LDS at the
// start, so that all of their loads are in flight together; then
//   diagonal V (DIAG): with v_u the diagonal of V_u,
//     D = HL rho + rho HR - sum_u ( v_u[i] (rho Lambda_u^+)[i][j] + (Lambda_u rho)[i][j] v_u[j] ),
//     HL = iH + sum_u V_u Lambda_u, HR = -iH + sum_u Lambda_u^+ V_u (formed at set-up),
//     read from LDS with no further barrier;
//   dense V: D = i[H, rho], then per noise T_u = Lambda_u rho - rho Lambda_u^+
//     into LDS, a barrier, and D += [V_u, T_u].
// LDS (cx<R> elements): rho, H or HL, HR (DIAG), per noise Lambda_u, Lambda_u^+
// and V_u (dense), then v_u (DIAG) or T (dense).
template <typename R, bool F64, int KP, Epi E, bool DIAG>
__global__ void __launch_bounds__(256) redfield_small_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  extern __shared__ __align__(16) unsigned char rf_lds[];
  C* sm = reinterpret_cast<C*>(rf_lds);
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const int N = d.N, N2 = d.N2, nn = d.n_noise;
  constexpr int per = DIAG ? 2 : 3;  // tables per noise
  C* s_rho = sm;
  C* s_H = sm + N2;  // H, or HL
  C* s_HR = sm + 2 * N2;
  C* s_tab = sm + 3 * N2;
  C* s_x = s_tab + static_cast<size_t>(per) * nn * N2;  // v_u (DIAG) or T (dense)
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const int e = threadIdx.x;
  const bool ok = e < N2;
  const int i = ok ? e / N : 0, j = ok ? e - (e / N) * N : 0;
  PreT<KP> pv;
  prefetch<F64, KP>(pv, A, cur, e, ok);
  for (int x = threadIdx.x; x < N2; x += blockDim.x) {
    s_rho[x] = in[x];
    s_H[x] = conv<R>(DIAG ? d.rf_HL[x] : d.H[x]);
    if (DIAG) s_HR[x] = conv<R>(d.rf_HR[x]);
  }
  for (int x = threadIdx.x; x < nn * N2; x += blockDim.x) {
    const int u = x / N2, y = x - u * N2;
    C* t = s_tab + static_cast<size_t>(u) * per * N2;
    t[y] = conv<R>(d.rf_L[x]);
    t[N2 + y] = conv<R>(d.rf_Ld[x]);
    if (!DIAG) t[2 * N2 + y] = conv<R>(d.V[x]);
  }
  if (DIAG)
    for (int x = threadIdx.x; x < nn * N; x += blockDim.x) s_x[x] = conv<R>(d.Vd[x]);
  __syncthreads();
  C D{0, 0};
  if (DIAG) {
    if (ok) {
      for (int k = 0; k < N; ++k) {
        cmac(D, s_H[i * N + k], s_rho[k * N + j]);
        cmac(D, s_rho[i * N + k], s_HR[k * N + j]);
      }
      for (int u = 0; u < nn; ++u) {
        const C* L = s_tab + static_cast<size_t>(u) * 2 * N2;
        const C* Ld = L + N2;
        C x{0, 0}, y{0, 0};
        for (int k = 0; k < N; ++k) {
          cmac(x, s_rho[i * N + k], Ld[k * N + j]);
          cmac(y, L[i * N + k], s_rho[k * N + j]);
        }
        const C vi = s_x[u * N + i], vj = s_x[u * N + j];
        cmac(D, C{-vi.re, -vi.im}, x);
        cmac(D, C{-vj.re, -vj.im}, y);
      }
    }
  } else {
    if (ok) {
      C c{0, 0};
      for (int k = 0; k < N; ++k) {
        cmac(c, s_H[i * N + k], s_rho[k * N + j]);
        cmac(c, s_rho[i * N + k], C{-s_H[k * N + j].re, -s_H[k * N + j].im});
      }
      D = times_i(c);
    }
    for (int u = 0; u < nn; ++u) {
      const C* L = s_tab + static_cast<size_t>(u) * 3 * N2;
      const C* Ld = L + N2;
      const C* V = L + 2 * N2;
      if (ok) {
        C t{0, 0};
        for (int k = 0; k < N; ++k) {
          cmac(t, L[i * N + k], s_rho[k * N + j]);
          cmac(t, s_rho[i * N + k], C{-Ld[k * N + j].re, -Ld[k * N + j].im});
        }
        s_x[e] = t;
      }
      __syncthreads();
      if (ok) {
        for (int k = 0; k < N; ++k) {
          cmac(D, V[i * N + k], s_x[k * N + j]);
          cmac(D, s_x[i * N + k], C{-V[k * N + j].re, -V[k * N + j].im});
        }
      }
      __syncthreads();
    }
  }
  double err = 0.0;
  if (ok) err = epilogue<F64, R, KP, E>(pv, A, cur, e, D, pg.alpha);
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, err);
}

// Larger problems, first pass: T_u = Lambda_u rho - rho Lambda_u^+ for every
// noise, one lane per (u, element); operands come through L1/L2.
template <typename R>
__global__ void __launch_bounds__(256) redfield_t_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const C* in = static_cast<const C*>(pick(A.in, pg.cur));
  C* T = static_cast<C*>(d.rf_T);
  const int N = d.N, N2 = d.N2;
  const long long total = static_cast<long long>(d.n_noise) * N2;
  for (long long x = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; x < total;
       x += static_cast<long long>(gridDim.x) * blockDim.x) {
    const long long u = x / N2;
    const int e = static_cast<int>(x - u * N2);
    const int i = e / N, j = e - i * N;
    const z128* L = d.rf_L + u * N2;
    const z128* Ld = d.rf_Ld + u * N2;
    C t{0, 0};
    for (int k = 0; k < N; ++k) {
      cmac(t, conv<R>(L[i * N + k]), in[k * N + j]);
      const C ld = conv<R>(Ld[k * N + j]);
      cmac(t, in[i * N + k], C{-ld.re, -ld.im});
    }
    T[x] = t;
  }
}

// Larger problems, second pass: D = i[H, rho] + sum_u [V_u, T_u] (diagonal V:
// (v_i - v_j) T_u[i][j]) and the stage epilogue, one lane per element.
template <typename R, bool F64, int KP, Epi E>
__global__ void __launch_bounds__(256) redfield_d_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const C* T = static_cast<const C*>(d.rf_T);
  const int N = d.N, N2 = d.N2;
  double err_acc = 0.0;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < N2; e += gridDim.x * blockDim.x) {
    PreT<KP> pv;
    prefetch<F64, KP>(pv, A, cur, e, true);
    const int i = e / N, j = e - i * N;
    C c{0, 0};
    for (int k = 0; k < N; ++k) {
      cmac(c, conv<R>(d.H[i * N + k]), in[k * N + j]);
      const C h = conv<R>(d.H[k * N + j]);
      cmac(c, in[i * N + k], C{-h.re, -h.im});
    }
    C D = times_i(c);
    for (int u = 0; u < d.n_noise; ++u) {
      const long long b = static_cast<long long>(u) * N2;
      if (d.diag_v) {
        cmac(D, conv<R>(d.Vd[u * N + i]) - conv<R>(d.Vd[u * N + j]), T[b + e]);
      } else {
        for (int k = 0; k < N; ++k) {
          cmac(D, conv<R>(d.V[b + i * N + k]), T[b + k * N + j]);
          const C v = conv<R>(d.V[b + k * N + j]);
          cmac(D, T[b + i * N + k], C{-v.re, -v.im});
        }
      }
    }
    err_acc += epilogue<F64, R, KP, E>(pv, A, cur, e, D, pg.alpha);
  }
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, err_acc);
}

// Sparse superoperator times the state, one 64-lane wavefront per row: the
// lanes stride over the row's entries (coalesced) and reduce with shuffles;
// lane 0 runs the epilogue.  Used for redfield_liou, whose rows hold up to
// N^2 entries (R = L - sum_u Phi_u Theta_u).
template <typename R, bool F64, int KP, Epi E>
__global__ void __launch_bounds__(256) csr_wave_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const int lane = threadIdx.x & 63;
  const long long wave = (static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const long long n_waves = (static_cast<long long>(gridDim.x) * blockDim.x) >> 6;
  double err_acc = 0.0;
  for (long long r = wave; r < d.main_size; r += n_waves) {
    PreT<KP> pv;
    prefetch<F64, KP>(pv, A, cur, r, lane == 0);
    C D{0, 0};
    for (long long p = d.R_ptr[r] + lane; p < d.R_ptr[r + 1]; p += 64)
      cmac(D, conv<R>(d.R_val[p]), in[d.R_col[p]]);
    for (int off = 32; off > 0; off >>= 1) {
      D.re += __shfl_down(D.re, off, 64);
      D.im += __shfl_down(D.im, off, 64);
    }
    if (lane == 0) err_acc += epilogue<F64, R, KP, E>(pv, A, cur, r, D, pg.alpha);
  }
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, err_acc);
}

}  // namespace

template <typename R, bool F64>
int launch_redfield(const FormDev& d, const StageArgs& A, hipStream_t st) {
  if (d.kind == HEOM_REDFIELD_LIOU) {
    const int grid = cap_grid((d.main_size + 3) / 4);  // four rows per workgroup
    with_epilogue<4, kMaxPre>(A, [&](auto kp, auto epi) {
      hipLaunchKernelGGL((csr_wave_kernel<R, F64, decltype(kp)::value, decltype(epi)::value>),
                         dim3(grid), dim3(256), 0, st, d, A);
    });
    return grid;
  }
  const bool diag = d.rf_HL != nullptr;
  const size_t lds = redfield_lds_elems(d.N2, d.N, d.n_noise, diag) * sizeof(cx<R>);
  if (d.N <= 16 && lds <= kRedfieldLds) {
    with_epilogue<4, kMaxPre>(A, [&](auto kp, auto epi) {
      constexpr int KP = decltype(kp)::value;
      constexpr Epi E = decltype(epi)::value;
      if (diag)
        hipLaunchKernelGGL((redfield_small_kernel<R, F64, KP, E, true>), dim3(1), dim3(256), lds,
                           st, d, A);
      else
        hipLaunchKernelGGL((redfield_small_kernel<R, F64, KP, E, false>), dim3(1), dim3(256), lds,
                           st, d, A);
    });
    return 1;
  }
  if (d.rf_T == nullptr) throw HeomError{HEOM_ERR_STATE, "redfield_hilb: scratch missing"};
  const long long nt = static_cast<long long>(d.n_noise) * d.N2;
  hipLaunchKernelGGL((redfield_t_kernel<R>), dim3(cap_grid((nt + 255) / 256)), dim3(256), 0, st,
                     d, A);
  const int grid = cap_grid((d.N2 + 255) / 256);
  with_epilogue<4, kMaxPre>(A, [&](auto kp, auto epi) {
    hipLaunchKernelGGL((redfield_d_kernel<R, F64, decltype(kp)::value, decltype(epi)::value>),
                       dim3(grid), dim3(256), 0, st, d, A);
  });
  return grid;
}

HAMD_FORM_INSTANCES(launch_redfield)

}  // namespace hamd
