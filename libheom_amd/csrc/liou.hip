// Superoperator forms: heom_liou, heom_ado and the Redfield QMEs.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// ---------------------------------------------------------------------------
// heom_liou: per-ADO superoperator form (heom_liou.h:151-255), N <= 16
// ---------------------------------------------------------------------------
template <typename R, bool F64, int KP>
__global__ void __launch_bounds__(256) liou_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  __shared__ C s_rho[256];
  __shared__ C s_phi[256];
  __shared__ C s_psi[256];
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const int N2 = d.N2;
  const int APB = 256 / N2;
  const int tid = threadIdx.x;
  const int la = tid / N2;
  const int e = tid - la * N2;
  const bool lane_ok = la < APB;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const int stride = N2 + 1;
  double err_acc = 0.0;
  const int n_groups = (d.n_hrchy + APB - 1) / APB;
  for (int g = blockIdx.x; g < n_groups; g += gridDim.x) {
    const int n = g * APB + la;
    const bool ok = lane_ok && n < d.n_hrchy;
    const long long gi = static_cast<long long>(n) * N2 + e;
    const C r = ok ? in[gi] : C{0, 0};
    PreT<KP> pv;
    prefetch<F64, KP>(pv, A, cur, gi, ok);
    if (lane_ok) s_rho[tid] = r;
    __syncthreads();
    C D{0, 0};
    int l0 = 0, l1 = 0;
    if (ok) {
      for (int p = d.sop_ptr[e]; p < d.sop_ptr[e + 1]; ++p)
        cmac(D, conv<R>(d.sop_val[p]), s_rho[la * N2 + d.sop_col[p]]);
      cmac(D, conv<R>(d.gam[n]), r);
      l0 = d.link_ptr[n];
      l1 = d.link_ptr[n + 1];
    }
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
      if (lane_ok) {
        s_phi[tid] = phi;
        s_psi[tid] = psi;
      }
      __syncthreads();
      if (ok) {
        const int* pp = d.sop_ptr + (1 + 2 * u) * stride;
        for (int p = pp[e]; p < pp[e + 1]; ++p)
          cmac(D, conv<R>(d.sop_val[p]), s_phi[la * N2 + d.sop_col[p]]);
        const int* pq = d.sop_ptr + (2 + 2 * u) * stride;
        for (int p = pq[e]; p < pq[e + 1]; ++p)
          cmac(D, conv<R>(d.sop_val[p]), s_psi[la * N2 + d.sop_col[p]]);
      }
      __syncthreads();
    }
    for (; l < l1; ++l) {
      const Link lk = d.links[l];
      const Coef c = d.coef[lk.cid];
      cmac(D, conv<R>(c.dir), in[static_cast<long long>(lk.nbr) * N2 + e]);
    }
    if (ok) err_acc += epilogue<F64, R, KP>(pv, A, cur, gi, D, pg.alpha);
    __syncthreads();
  }
  if (A.do_err) write_partial(A, err_acc);
}

// heom_liou for 16 < N <= 32 (N^2 up to 1024): one ADO per 256-lane workgroup,
// each lane up to four elements e = tid + 256 c, rho_n and the per-noise
// neighbour sums phi, psi staged in LDS (3 N^2 complex values, dynamic);
// the same per-element operation order as liou_kernel.
template <typename R, bool F64, int KP>
__global__ void __launch_bounds__(256) liou_wide_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  constexpr int NC = 4;
  extern __shared__ __align__(16) unsigned char s_dyn[];
  const int N2 = d.N2;
  C* s_rho = reinterpret_cast<C*>(s_dyn);
  C* s_phi = s_rho + N2;
  C* s_psi = s_phi + N2;
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const int tid = threadIdx.x;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const int stride = N2 + 1;
  double err_acc = 0.0;
  for (int n = blockIdx.x; n < d.n_hrchy; n += gridDim.x) {
    const long long base = static_cast<long long>(n) * N2;
    for (int e = tid; e < N2; e += 256) s_rho[e] = in[base + e];
    __syncthreads();
    C D[NC];
    const C gm = conv<R>(d.gam[n]);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int e = tid + 256 * c;
      D[c] = C{0, 0};
      if (e < N2) {
        for (int p = d.sop_ptr[e]; p < d.sop_ptr[e + 1]; ++p)
          cmac(D[c], conv<R>(d.sop_val[p]), s_rho[d.sop_col[p]]);
        cmac(D[c], gm, s_rho[e]);
      }
    }
    const int l1 = d.link_ptr[n + 1];
    int l = d.link_ptr[n];
    for (int u = 0; u < d.n_noise; ++u) {
      C phi[NC], psi[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) phi[c] = psi[c] = C{0, 0};
      while (l < l1) {
        const Link lk = d.links[l];
        const Coef cf = d.coef[lk.cid];
        if (cf.u != u) break;
        const C* nb = in + static_cast<long long>(lk.nbr) * N2;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int e = tid + 256 * c;
          if (e < N2) {
            const C x = nb[e];
            cmac(phi[c], conv<R>(cf.phi), x);
            cmac(psi[c], conv<R>(cf.psi), x);
          }
        }
        ++l;
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int e = tid + 256 * c;
        if (e < N2) {
          s_phi[e] = phi[c];
          s_psi[e] = psi[c];
        }
      }
      __syncthreads();
      const int* pp = d.sop_ptr + (1 + 2 * u) * stride;
      const int* pq = d.sop_ptr + (2 + 2 * u) * stride;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int e = tid + 256 * c;
        if (e < N2) {
          for (int p = pp[e]; p < pp[e + 1]; ++p)
            cmac(D[c], conv<R>(d.sop_val[p]), s_phi[d.sop_col[p]]);
          for (int p = pq[e]; p < pq[e + 1]; ++p)
            cmac(D[c], conv<R>(d.sop_val[p]), s_psi[d.sop_col[p]]);
        }
      }
      __syncthreads();
    }
    for (; l < l1; ++l) {
      const Link lk = d.links[l];
      const Coef cf = d.coef[lk.cid];
      const C* nb = in + static_cast<long long>(lk.nbr) * N2;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int e = tid + 256 * c;
        if (e < N2) cmac(D[c], conv<R>(cf.dir), nb[e]);
      }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int e = tid + 256 * c;
      if (e < N2) {
        PreT<KP> pv;
        prefetch<F64, KP>(pv, A, cur, base + e, true);
        err_acc += epilogue<F64, R, KP>(pv, A, cur, base + e, D[c], pg.alpha);
      }
    }
    __syncthreads();
  }
  if (A.do_err) write_partial(A, err_acc);
}

// ---------------------------------------------------------------------------
// heom_ado: one global CSR matrix-vector product (heom_ado.h:191-202)
// ---------------------------------------------------------------------------
template <typename R, bool F64, int KP>
__global__ void __launch_bounds__(256) ado_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  double err_acc = 0.0;
  const long long rows = d.main_size;
  for (long long r = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; r < rows;
       r += static_cast<long long>(gridDim.x) * blockDim.x) {
    PreT<KP> pv;
    prefetch<F64, KP>(pv, A, cur, r, true);
    C D{0, 0};
    for (long long p = d.R_ptr[r]; p < d.R_ptr[r + 1]; ++p)
      cmac(D, conv<R>(d.R_val[p]), in[d.R_col[p]]);
    err_acc += epilogue<F64, R, KP>(pv, A, cur, r, D, pg.alpha);
  }
  if (A.do_err) write_partial(A, err_acc);
}

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
template <typename R, bool F64, int KP, bool DIAG>
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
  if (ok) err = epilogue<F64, R, KP>(pv, A, cur, e, D, pg.alpha);
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
template <typename R, bool F64, int KP>
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
    err_acc += epilogue<F64, R, KP>(pv, A, cur, e, D, pg.alpha);
  }
  if (A.do_err) write_partial(A, err_acc);
}

// Sparse superoperator times the state, one 64-lane wavefront per row: the
// lanes stride over the row's entries (coalesced) and reduce with shuffles;
// lane 0 runs the epilogue.  Used for redfield_liou, whose rows hold up to
// N^2 entries (R = L - sum_u Phi_u Theta_u).
template <typename R, bool F64, int KP>
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
    if (lane == 0) err_acc += epilogue<F64, R, KP>(pv, A, cur, r, D, pg.alpha);
  }
  if (A.do_err) write_partial(A, err_acc);
}

}  // namespace

template <typename R, bool F64>
int launch_liou(const FormDev& d, const StageArgs& A, hipStream_t st) {
  if (d.N2 > 256) {
    // 16 < N <= 32: one ADO per workgroup (set_param refuses larger N)
    const int grid = cap_grid(d.n_hrchy);
    const size_t lds = 3 * sizeof(cx<R>) * static_cast<size_t>(d.N2);
    if (A.npre <= 4)
      hipLaunchKernelGGL((liou_wide_kernel<R, F64, 4>), dim3(grid), dim3(256), lds, st, d, A);
    else
      hipLaunchKernelGGL((liou_wide_kernel<R, F64, kMaxPre>), dim3(grid), dim3(256), lds, st, d,
                         A);
    return grid;
  }
  const int APB = 256 / d.N2;
  const int grid = cap_grid((d.n_hrchy + APB - 1) / APB);
  if (A.npre <= 4)
    hipLaunchKernelGGL((liou_kernel<R, F64, 4>), dim3(grid), dim3(256), 0, st, d, A);
  else
    hipLaunchKernelGGL((liou_kernel<R, F64, kMaxPre>), dim3(grid), dim3(256), 0, st, d, A);
  return grid;
}

template <typename R, bool F64>
int launch_ado(const FormDev& d, const StageArgs& A, hipStream_t st) {
  const int grid = cap_grid((d.main_size + 255) / 256);
  if (A.npre <= 4)
    hipLaunchKernelGGL((ado_kernel<R, F64, 4>), dim3(grid), dim3(256), 0, st, d, A);
  else
    hipLaunchKernelGGL((ado_kernel<R, F64, kMaxPre>), dim3(grid), dim3(256), 0, st, d, A);
  return grid;
}

template <typename R, bool F64>
int launch_redfield(const FormDev& d, const StageArgs& A, hipStream_t st) {
  const bool small = A.npre <= 4;
  if (d.kind == HEOM_REDFIELD_LIOU) {
    const int grid = cap_grid((d.main_size + 3) / 4);  // four rows per workgroup
    if (small)
      hipLaunchKernelGGL((csr_wave_kernel<R, F64, 4>), dim3(grid), dim3(256), 0, st, d, A);
    else
      hipLaunchKernelGGL((csr_wave_kernel<R, F64, kMaxPre>), dim3(grid), dim3(256), 0, st, d, A);
    return grid;
  }
  const bool diag = d.rf_HL != nullptr;
  const size_t lds = redfield_lds_elems(d.N2, d.N, d.n_noise, diag) * sizeof(cx<R>);
  if (d.N <= 16 && lds <= kRedfieldLds) {
#define HAMD_RF(DG, KPV)                                                                    \
  hipLaunchKernelGGL((redfield_small_kernel<R, F64, KPV, DG>), dim3(1), dim3(256), lds, st, d, \
                     A)
    if (diag) {
      if (small) HAMD_RF(true, 4); else HAMD_RF(true, kMaxPre);
    } else {
      if (small) HAMD_RF(false, 4); else HAMD_RF(false, kMaxPre);
    }
#undef HAMD_RF
    return 1;
  }
  if (d.rf_T == nullptr) throw HeomError{HEOM_ERR_STATE, "redfield_hilb: scratch missing"};
  const long long nt = static_cast<long long>(d.n_noise) * d.N2;
  hipLaunchKernelGGL((redfield_t_kernel<R>), dim3(cap_grid((nt + 255) / 256)), dim3(256), 0, st,
                     d, A);
  const int grid = cap_grid((d.N2 + 255) / 256);
  if (small)
    hipLaunchKernelGGL((redfield_d_kernel<R, F64, 4>), dim3(grid), dim3(256), 0, st, d, A);
  else
    hipLaunchKernelGGL((redfield_d_kernel<R, F64, kMaxPre>), dim3(grid), dim3(256), 0, st, d, A);
  return grid;
}

HAMD_FORM_INSTANCES(launch_liou)
HAMD_FORM_INSTANCES(launch_ado)
HAMD_FORM_INSTANCES(launch_redfield)

}  // namespace hamd
