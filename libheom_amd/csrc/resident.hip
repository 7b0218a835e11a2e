// Resident integrators: whole solves of small problems in one workgroup.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// ---------------------------------------------------------------------------
// Resident fixed-step integrator: heom_hilb with diagonal V, FP64, at most
// kResidentMax elements.  One workgroup keeps the state and every stage buffer
// in LDS and runs all steps of an output interval; one lane per element.  The
// per-element link coefficients (neighbour element, c = cm*i*phi + ac*psi +
// dir, the same expression the fast kernel forms per stage) and Gamma_n +
// delta term are computed once into registers.  Stage arithmetic follows the
// epilogue of the stage kernels (k = -dt*D, sum of c_s*operand_s then + ck*k).
// ---------------------------------------------------------------------------
// One lane's element of a resident problem: the link coefficients and
// neighbour elements (computed once) and the operator D at that element.
// NS: the number of levels (0: any); KH (two levels): the lane keeps its row and
// column of H.
template <int MAXL, int NS, bool KH = false>
struct ResidentElem {
  int g, i, j, nl;
  z128 diag;
  int nbr[MAXL];
  z128 cf[MAXL];
  z128 hr[KH ? 2 : 1], hc[KH ? 2 : 1];

  __device__ __forceinline__ void init(const FormDev& d, int e, bool ok) {
    const int N = d.N, N2 = d.N2;
    g = ok ? e / N2 : 0;
    const int ee = ok ? e - g * N2 : 0;
    i = ee / N;
    j = ee - (ee / N) * N;
    const int l0 = d.link_ptr[g], l1 = d.link_ptr[g + 1];
    nl = ok ? l1 - l0 : 0;
    diag = d.gam[g] + d.dterm[ee];
    if constexpr (KH) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        hr[k] = d.H[i * 2 + k];
        hc[k] = d.H[k * 2 + j];
      }
    }
#pragma unroll
    for (int l = 0; l < MAXL; ++l) {
      nbr[l] = 0;
      cf[l] = z128{0.0, 0.0};
      if (l < nl) {
        const LinkFlat q = d.flat[l0 + l];
        nbr[l] = q.nbr * N2 + ee;
        const long long b = static_cast<long long>(q.u) * N2 + ee;
        if (d.real_v) {
          const z128 p = d.cmac_tab[b];
          cf[l].re = p.re * q.iphi.re + p.im * q.psi.re + q.dir.re;
          cf[l].im = p.re * q.iphi.im + p.im * q.psi.im + q.dir.im;
        } else {
          cf[l] = d.cmac_tab[2 * b] * q.iphi + d.cmac_tab[2 * b + 1] * q.psi + q.dir;
        }
      }
    }
  }

  // LDS table: H
  static __host__ __device__ size_t tab_elems(int N, int n_noise) { return static_cast<size_t>(N) * N; }
  static __device__ __forceinline__ void stage(const FormDev& d, z128* tab) {
    for (int x = threadIdx.x; x < d.N2; x += blockDim.x) tab[x] = d.H[x];
  }

  // D at element e of the state X, x its own element (same expression order as
  // the stage kernels).  AHEAD: every neighbour's load before the first product
  template <bool AHEAD>
  __device__ __forceinline__ z128 op(const z128* X, const z128* s_H, z128 x, int n, int n2) const {
    const int N = NS ? NS : n, N2 = NS ? NS * NS : n2;
    const z128* Xg = X + static_cast<size_t>(g) * N2;
    z128 xn[MAXL];
    if constexpr (AHEAD) {
#pragma unroll
      for (int l = 0; l < MAXL; ++l)
        if (l < nl) xn[l] = X[nbr[l]];
    }
    z128 acc{0.0, 0.0};
    constexpr int U = NS ? NS : 1;
#pragma unroll U
    for (int k = 0; k < N; ++k) {
      z128 h0, h1;
      if constexpr (KH) {
        h0 = hr[k];
        h1 = hc[k];
      } else {
        h0 = s_H[i * N + k];
        h1 = s_H[k * N + j];
      }
      cmac(acc, h0, Xg[k * N + j]);
      const z128 t = Xg[i * N + k];
      cmac(acc, z128{-t.re, -t.im}, h1);
    }
    z128 D = times_i(acc);
    cmac(D, diag, x);
#pragma unroll
    for (int l = 0; l < MAXL; ++l)
      if (l < nl) {
        // the product that is not rounded is the one of the stage kernels, whose bits
        // a fixed-step solve with real parameters keeps
        const z128 c = cf[l], v = AHEAD ? xn[l] : X[nbr[l]];
        D.re += fma(c.re, v.re, -(c.im * v.im));
        D.im += fma(c.im, v.re, c.re * v.im);
      }
    return D;
  }
};

// One element of a resident redfield_hilb problem with diagonal V: the
// operator of redfield_small_kernel<..., true> (D = HL rho + rho HR -
// sum_u (v_u[i] (rho Lambda_u^+)[i][j] + (Lambda_u rho)[i][j] v_u[j])), same
// expression order, with its tables in LDS.
struct RedfieldElem {
  int i, j, nn;
  // LDS table: HL, HR, per noise Lambda_u and Lambda_u^+, then v_u (n_noise x N)
  static __host__ __device__ size_t tab_elems(int N, int n_noise) {
    return static_cast<size_t>(2 + 2 * n_noise) * N * N + static_cast<size_t>(n_noise) * N;
  }
  static __device__ __forceinline__ void stage(const FormDev& d, z128* tab) {
    const int N2 = d.N2, nn = d.n_noise;
    for (int x = threadIdx.x; x < N2; x += blockDim.x) {
      tab[x] = d.rf_HL[x];
      tab[N2 + x] = d.rf_HR[x];
    }
    for (int x = threadIdx.x; x < nn * N2; x += blockDim.x) {
      const int u = x / N2, y = x - u * N2;
      tab[static_cast<size_t>(2 + 2 * u) * N2 + y] = d.rf_L[x];
      tab[static_cast<size_t>(3 + 2 * u) * N2 + y] = d.rf_Ld[x];
    }
    for (int x = threadIdx.x; x < nn * d.N; x += blockDim.x)
      tab[static_cast<size_t>(2 + 2 * nn) * N2 + x] = d.Vd[x];
  }
  __device__ __forceinline__ void init(const FormDev& d, int e, bool ok) {
    const int ee = ok ? e : 0;
    i = ee / d.N;
    j = ee - i * d.N;
    nn = d.n_noise;
  }
  template <bool>
  __device__ __forceinline__ z128 op(const z128* X, const z128* tab, z128, int N, int N2) const {
    const z128* HL = tab;
    const z128* HR = tab + N2;
    z128 D{0.0, 0.0};
    for (int k = 0; k < N; ++k) {
      cmac(D, HL[i * N + k], X[k * N + j]);
      cmac(D, X[i * N + k], HR[k * N + j]);
    }
    const z128* v = tab + static_cast<size_t>(2 + 2 * nn) * N2;
    for (int u = 0; u < nn; ++u) {
      const z128* L = tab + static_cast<size_t>(2 + 2 * u) * N2;
      const z128* Ld = L + N2;
      z128 x{0.0, 0.0}, y{0.0, 0.0};
      for (int k = 0; k < N; ++k) {
        cmac(x, X[i * N + k], Ld[k * N + j]);
        cmac(y, L[i * N + k], X[k * N + j]);
      }
      const z128 vi = v[u * N + i], vj = v[u * N + j];
      cmac(D, z128{-vi.re, -vi.im}, x);
      cmac(D, z128{-vj.re, -vj.im}, y);
    }
    return D;
  }
};

// LDS buffers of a stage program: one for each slot that some stage reads as
// its operator input; every other operand stays in the lane's registers.
constexpr int res_buf(const ResidentProg& P, int slot) {
  int n = 0;
  for (int q = 0; q < P.n_buf; ++q) {
    bool in = false;
    for (int s = 0; s < P.n_stages; ++s) in = in || P.st[s].in == q;
    if (q == slot) return in ? n : -1;
    n += in ? 1 : 0;
  }
  return -1;
}

// The results to the host: every lane's element is in host memory before the
// progress word is.
__device__ __forceinline__ void post_host(const ResidentHost& h, bool ok, int e, z128 y) {
  if (h.mail == nullptr) return;
  if (ok) h.y[e] = y;
  __threadfence_system();
  __syncthreads();
  if (e == 0)
    __hip_atomic_store(h.mail, 1ull << 2, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// What bounds it: one workgroup, a barrier per stage, and between two barriers
// the LDS reads (own row and column, up to MAXL neighbours), the chain of FP64
// sums and one LDS write.  With the level count compiled in and every operand
// but the stage input in registers a stage of the 264-element spin-boson
// hierarchy takes 0.47 us (0.58 us with rolled loops and all operands in LDS);
// what is left is FP64 issue: some 80 instructions of 4 cycles per wavefront, two
// wavefronts on one SIMD.
template <class E, int SCHEME, int BS>
__global__ void __launch_bounds__(BS) resident_kernel(const FormDev d, const ResidentArgs a) {
  extern __shared__ __align__(16) unsigned char res_lds[];
  constexpr const ResidentProg& P = SCHEME == 1 ? kResidentRk4 : kResidentLsrk4;
  z128* buf = reinterpret_cast<z128*>(res_lds);
  const int ms = static_cast<int>(d.main_size);
  const int N = d.N, N2 = d.N2;
  z128* s_H = buf + static_cast<size_t>(P.n_buf) * ms;  // the element type's tables
  const int e = threadIdx.x;
  const bool ok = e < ms;
  z128 r[4];  // the lane's element of every slot; slot 0: the state
  r[0] = ok ? a.y[e] : z128{0.0, 0.0};
  r[1] = r[2] = r[3] = z128{0.0, 0.0};
  if (ok) buf[e] = r[0];
  E::stage(d, s_H);
  E el;
  el.init(d, e, ok);
  __syncthreads();
  const int n_int = a.n_int > 0 ? a.n_int : 1;
  for (int iv = 0; iv < n_int; ++iv) {
    const long long n_full = a.n_int > 0 ? a.n_full_i[iv] : a.n_full;
    const double dt_last = a.n_int > 0 ? a.dt_last_i[iv] : a.dt_last;
    if (a.n_int > 0 && e < N2) a.rho_s[static_cast<size_t>(iv) * N2 + e] = r[0];
    const long long n_steps = n_full + 1;
    for (long long step = 0; step < n_steps; ++step) {
      const double dt = step < n_full ? a.dt : dt_last;
#pragma unroll
      for (int s = 0; s < P.n_stages; ++s) {
        if (ok) {
          const z128 D = el.template op<BS <= 512>(
              buf + static_cast<size_t>(res_buf(P, P.st[s].in)) * ms, s_H,
              r[P.st[s].in], N, N2);
          const z128 k{-(dt * D.re - 0.0 * D.im), -(dt * D.im + 0.0 * D.re)};
          z128 v[2];
#pragma unroll
          for (int c = 0; c < P.st[s].ncombo; ++c) {
            v[c] = z128{0.0, 0.0};
#pragma unroll
            for (int p = 0; p < P.st[s].npre; ++p) {
              v[c].re = fma(P.st[s].cc[c][p], r[P.st[s].pre[p]].re, v[c].re);
              v[c].im = fma(P.st[s].cc[c][p], r[P.st[s].pre[p]].im, v[c].im);
            }
            v[c].re = fma(P.st[s].ck[c], k.re, v[c].re);
            v[c].im = fma(P.st[s].ck[c], k.im, v[c].im);
          }
#pragma unroll
          for (int c = 0; c < P.st[s].ncombo; ++c) {
            const int dst = P.st[s].dst[c];
            r[dst] = v[c];
            if (res_buf(P, dst) >= 0) buf[static_cast<size_t>(res_buf(P, dst)) * ms + e] = v[c];
          }
        }
        __syncthreads();
      }
    }
  }
  if (a.n_int > 0 && e < N2) a.rho_s[static_cast<size_t>(a.n_int) * N2 + e] = r[0];
  if (ok) a.y[e] = r[0];
  post_host(a.host, ok, e, r[0]);
}

// Resident Dormand-Prince: the adaptive solve of a small heom_hilb problem
// (diagonal V, FP64) in one workgroup.  Stage arithmetic follows the stage
// kernels (k = -dt*D; y + sum a_ij k_j as one fma chain in operand order; the
// error combination and weights of rkdp.h:136-153) and each output interval
// starts as ctrl_init_kernel does.  Up to 512 elements, where a lane has 256
// registers, y, y_new and k1..k6 stay in registers; LDS holds the operator
// inputs: 0/1 the y / y_new pair (swapped on acceptance), 2/3 the stage inputs,
// and 4..9 the lanes' own k's of the larger problems.  The error norm is summed in a
// fixed order: wavefront shuffles, then the waves, one after another, or with a.tree as
// dopri_step_kernel adds up to sixteen partials of one-wave workgroups (lane w of its
// first wavefront holds partial w): a change there has to be made here.  Up to eight
// wavefronts every lane runs the step control on it (no round trip through LDS);
// with more, lane 0 does (all sixteen wavefronts computing the power of the error
// took 20% of a solve).
template <class E, int BS>
__global__ void __launch_bounds__(BS)
    resident_dopri_kernel(const FormDev d, const ResidentDopriArgs a) {
  extern __shared__ __align__(16) unsigned char res_lds[];
  __shared__ double s_red[16];
  __shared__ Ctrl s_c;
  z128* buf = reinterpret_cast<z128*>(res_lds);
  const int ms = static_cast<int>(d.main_size);
  const int N = d.N, N2 = d.N2;
  z128* s_H = buf + static_cast<size_t>(kResidentDopriBuf) * ms;
  const int e = threadIdx.x;
  const bool ok = e < ms;
  z128 y = ok ? a.y[e] : z128{0.0, 0.0};
  if (ok) buf[e] = y;
  if (e < 16) s_red[e] = 0.0;
  E::stage(d, s_H);
  E el;
  el.init(d, e, ok);
  // the control block: in the lane's registers, or (beyond 512 elements) in LDS
  // and written by lane 0
  constexpr bool REG = BS <= 512;
  Ctrl c_reg;
  Ctrl& c = REG ? c_reg : s_c;
  const bool owner = REG || e == 0;
  if (owner) {
    c = Ctrl{};
    c.dt = a.dt_first;
  }
  int gave_up = 0;
  __syncthreads();
  if (a.rho_s && e < N2) a.rho_s[e] = y;
  z128* SA = buf + 2 * static_cast<size_t>(ms);
  z128* SB = buf + 3 * static_cast<size_t>(ms);
  z128* KL = buf + 4 * static_cast<size_t>(ms);  // k1..k6 beyond 512 elements
  // D of the current state: the first evaluation of an attempt is the last one of
  // the attempt that produced the state (a rejected one keeps its own)
  z128 dy{0.0, 0.0};
  if (ok) dy = el.template op<REG>(buf, s_H, y, N, N2);
  for (int iv = 0; iv < a.n_int; ++iv) {
    // ctrl_init_kernel: dt carries over from the last attempt
    const double t0 = a.t_list ? a.t_list[iv] : a.t0, t1 = a.t_list ? a.t_list[iv + 1] : a.t1;
    if (owner) {
      c.t = t0;
      c.t_bound = t1;
      c.count = 1;
      c.gave_up = 0;
      // a zero-length interval takes no attempt and keeps the step size
      c.done = (t1 > t0) ? 0 : 1;
      if (!c.done && t0 + c.dt > t1) c.dt = t1 - t0;
    }
    if (!REG) __syncthreads();
    while (!c.done) {
      const double dt = c.dt;
      const int cur = c.cur;
      const z128* Y = buf + (cur ? ms : 0);
      z128* YN = buf + (cur ? 0 : ms);
      z128 Kr[REG ? 6 : 1], x = y;  // x (REG): the stage input of the lane's element
      auto K = [&](int j) -> z128& {
        if constexpr (REG)
          return Kr[j];
        else
          return KL[static_cast<size_t>(j) * ms + e];
      };
#pragma unroll
      for (int st = 0; st < 6; ++st) {
        const z128* in = st == 0 ? Y : ((st & 1) ? SA : SB);
        z128* out = st == 5 ? YN : ((st & 1) ? SB : SA);
        if (ok) {
          const z128 D =
              st == 0 ? dy : el.template op<REG>(in, s_H, REG ? x : in[e], N, N2);
          const z128 k{-(dt * D.re - 0.0 * D.im), -(dt * D.im + 0.0 * D.re)};
          K(st) = k;
          const z128 y0 = REG ? y : Y[e];
          z128 v{fma(1.0, y0.re, 0.0), fma(1.0, y0.im, 0.0)};
#pragma unroll
          for (int j = 0; j < st; ++j) {
            const double w = st < 5 ? kDpA[st + 1][j] : kDpB[j];
            if (st < 5 || w != 0.0) {
              const z128 kj = K(j);
              v.re = fma(w, kj.re, v.re);
              v.im = fma(w, kj.im, v.im);
            }
          }
          const double w = st < 5 ? kDpA[st + 1][st] : kDpB[5];
          v.re = fma(w, k.re, v.re);
          v.im = fma(w, k.im, v.im);
          out[e] = v;
          if (REG) x = v;
        }
        __syncthreads();
      }
      double w2 = 0.0;
      z128 D{0.0, 0.0};
      if (ok) {
        const z128 yn = REG ? x : YN[e], yo = REG ? y : Y[e];
        D = el.template op<REG>(YN, s_H, yn, N, N2);
        const z128 k{-(dt * D.re - 0.0 * D.im), -(dt * D.im + 0.0 * D.re)};
        z128 er{0.0, 0.0};
#pragma unroll
        for (int j = 0; j < 6; ++j) {
          if (kDpE[j] != 0.0) {
            const z128 kj = K(j);
            er.re = fma(kDpE[j], kj.re, er.re);
            er.im = fma(kDpE[j], kj.im, er.im);
          }
        }
        // the stage kernels' padded sixth operand adds 0*0
        er.re = fma(0.0, 0.0, er.re);
        er.im = fma(0.0, 0.0, er.im);
        er.re = fma(kDpE[6], k.re, er.re);
        er.im = fma(kDpE[6], k.im, er.im);
        // |z| with the fma on the part that the stage kernels put it on (a.tree),
        // so that the norm is theirs to the last bit
        const double a1 = sqrt(fma(yn.re, yn.re, yn.im * yn.im));
        const double a0 = sqrt(fma(yo.re, yo.re, yo.im * yo.im));
        const double e2 = a.tree ? fma(er.im, er.im, er.re * er.re)
                                 : fma(er.re, er.re, er.im * er.im);
        const double w = sqrt(e2) / (a.atol + a.rtol * (a1 > a0 ? a1 : a0));
        w2 = w * w;
      }
      for (int off = 32; off > 0; off >>= 1) w2 += __shfl_down(w2, off, 64);
      if ((e & 63) == 0) s_red[e >> 6] = w2;
      __syncthreads();
      // (the next write to s_red comes six barriers later)
      if (owner) {
        double t = 0.0;
        if (a.tree) {
          // the 16-lane shuffle tree; rolled, its operands would take 32 registers
          double c0 = 0.0, c1 = 0.0;
#pragma unroll 1
          for (int w = 0; w < 4; ++w) {
            const double b = (s_red[w] + s_red[w + 8]) + (s_red[w + 4] + s_red[w + 12]);
            if (w & 1)
              c1 += b;
            else
              c0 += b;
          }
          t = c0 + c1;
        } else {
          for (int w = 0; w < static_cast<int>(blockDim.x >> 6); ++w) t += s_red[w];
        }
        dopri_control(&c, sqrt(t * a.inv_n));
      }
      if (!REG) __syncthreads();
      if (c.gave_up) gave_up = 1;
      if (c.cur != cur) {
        dy = D;
        if (REG) y = x;
      }
    }
    if (!REG && ok) y = buf[(c.cur ? ms : 0) + e];
    if (a.rho_s && e < N2) a.rho_s[static_cast<size_t>(iv + 1) * N2 + e] = y;
    // every wave has read the control block before lane 0 starts the next interval
    if (!REG) __syncthreads();
  }
  if (ok) a.y[e] = y;
  if (e == 0) {
    Ctrl out = c;
    out.gave_up = gave_up;
    *a.ctrl = out;
    if (a.host.mail) *a.host.ctrl = out;
  }
  post_host(a.host, ok, e, y);
}

}  // namespace

bool resident_ok(const FormDev& d, int max_links) {
  if (d.main_size > kResidentMax || d.clos != nullptr) return false;
  if (d.kind == HEOM_HILB) return d.diag_v && max_links <= 8;
  return d.kind == HEOM_REDFIELD_HILB && d.rf_HL != nullptr;  // diagonal V
}

namespace {
size_t resident_tab_elems(const FormDev& d) {
  return d.kind == HEOM_REDFIELD_HILB ? RedfieldElem::tab_elems(d.N, d.n_noise)
                                      : ResidentElem<4, 0>::tab_elems(d.N, d.n_noise);
}
}  // namespace

size_t resident_lds_bytes(const FormDev& d, int n_buf) {
  return sizeof(z128) * (static_cast<size_t>(n_buf) * d.main_size + resident_tab_elems(d));
}

namespace {
// f(element type tag) for the problem's element type
template <class E>
struct Tag {
  using type = E;
};
template <int MAXL, bool KH, class F>
void with_levels(int N, F f) {
  if (N == 2) return f(Tag<ResidentElem<MAXL, 2, KH>>{});
  if (N == 4) return f(Tag<ResidentElem<MAXL, 4>>{});
  return f(Tag<ResidentElem<MAXL, 0>>{});
}
template <bool KH, class F>
void with_elem(const FormDev& d, int max_links, F f) {
  if (d.kind == HEOM_REDFIELD_HILB) return f(Tag<RedfieldElem>{});
  if (max_links <= 4) return with_levels<4, KH>(d.N, f);
  if (max_links <= 6) return with_levels<6, KH>(d.N, f);
  return with_levels<8, KH>(d.N, f);
}

template <class E, int SCHEME, int BS>
void launch_resident_as(const FormDev& d, const ResidentArgs& a, int bs, size_t lds,
                        hipStream_t st) {
  static bool once = (allow_lds(resident_kernel<E, SCHEME, BS>, kResidentLds), true);
  (void)once;
  hipLaunchKernelGGL((resident_kernel<E, SCHEME, BS>), dim3(1), dim3(bs), lds, st, d, a);
}

template <class E, int BS>
void launch_resident_dopri_as(const FormDev& d, const ResidentDopriArgs& a, int bs, size_t lds,
                              hipStream_t st) {
  static bool once = (allow_lds(resident_dopri_kernel<E, BS>, kResidentLds), true);
  (void)once;
  hipLaunchKernelGGL((resident_dopri_kernel<E, BS>), dim3(1), dim3(bs), lds, st, d, a);
}
}  // namespace

// Up to 512 elements a lane may use 256 registers, beyond 128.
void launch_resident(const FormDev& d, int max_links, const ResidentArgs& a, hipStream_t stream) {
  const int ms = static_cast<int>(d.main_size);
  if (!resident_ok(d, max_links) || (a.scheme != 1 && a.scheme != 2))
    throw HeomError{HEOM_ERR_STATE, "resident integrator: unsupported problem"};
  const int n_buf = a.scheme == 1 ? kResidentRk4.n_buf : kResidentLsrk4.n_buf;
  const size_t lds = resident_lds_bytes(d, n_buf);
  if (lds > kResidentLds) throw HeomError{HEOM_ERR_STATE, "resident integrator: LDS exceeded"};
  const int bs = ((ms + 63) / 64) * 64;
  if (bs <= 512) {
    with_elem<true>(d, max_links, [&](auto tag) {
      using E = typename decltype(tag)::type;
      if (a.scheme == 1)
        launch_resident_as<E, 1, 512>(d, a, bs, lds, stream);
      else
        launch_resident_as<E, 2, 512>(d, a, bs, lds, stream);
    });
  } else {
    with_elem<false>(d, max_links, [&](auto tag) {
      using E = typename decltype(tag)::type;
      if (a.scheme == 1)
        launch_resident_as<E, 1, 1024>(d, a, bs, lds, stream);
      else
        launch_resident_as<E, 2, 1024>(d, a, bs, lds, stream);
    });
  }
  HAMD_HIP(hipGetLastError());
}

bool resident_dopri_ok(const FormDev& d, int max_links) {
  return resident_ok(d, max_links) && d.main_size <= kResidentDopriMax &&
         resident_lds_bytes(d, kResidentDopriBuf) <= kResidentLds;
}

void launch_resident_dopri(const FormDev& d, int max_links, const ResidentDopriArgs& a,
                           hipStream_t stream) {
  if (!resident_dopri_ok(d, max_links) || a.n_int < 1)
    throw HeomError{HEOM_ERR_STATE, "resident Dormand-Prince: unsupported problem"};
  const int ms = static_cast<int>(d.main_size);
  const size_t lds = resident_lds_bytes(d, kResidentDopriBuf);
  if (lds > kResidentLds) throw HeomError{HEOM_ERR_STATE, "resident Dormand-Prince: LDS exceeded"};
  const int bs = ((ms + 63) / 64) * 64;
  if (bs <= 512)
    with_elem<true>(d, max_links, [&](auto tag) {
      launch_resident_dopri_as<typename decltype(tag)::type, 512>(d, a, bs, lds, stream);
    });
  else
    with_elem<false>(d, max_links, [&](auto tag) {
      launch_resident_dopri_as<typename decltype(tag)::type, 1024>(d, a, bs, lds, stream);
    });
  HAMD_HIP(hipGetLastError());
}

}  // namespace hamd
