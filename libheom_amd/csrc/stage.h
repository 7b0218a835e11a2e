// Device code shared by the operator kernels: operand loads and stores, the
// Runge-Kutta epilogue, the kernel prologue, error-norm partials and the
// Dormand-Prince step control.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "../../include/libheom_amd.h"
#include "common.h"
#include "kernels.h"

namespace hamd {

namespace {

typedef float mf_f4 __attribute__((ext_vector_type(4)));  // f32 matrix-core accumulator

// read-only tables through the constant address space: uniform indices then
// compile to scalar loads
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* cst(const T* p) {
  return (const __attribute__((address_space(4))) T*)(p);
}

template <typename T>
using cptr = const __attribute__((address_space(4))) T*;

__device__ __forceinline__ LinkFlat ld_flat(cptr<LinkFlat> p) {
  LinkFlat f;
  f.nbr = p->nbr;
  f.u = p->u;
  f.iphi = z128{p->iphi.re, p->iphi.im};
  f.psi = z128{p->psi.re, p->psi.im};
  f.dir = z128{p->dir.re, p->dir.im};
  return f;
}

// Link l from the 8-byte record (neighbour, coefficient index) and its entry in
// the hierarchy's deduplicated coefficient table (one entry per mode,
// occupation and direction: a few KB, held by the scalar cache); i*phi is
// formed exactly (a swap and a negation), as the host does for LinkFlat.
__device__ __forceinline__ LinkFlat ld_link_coef(cptr<Link> lk, cptr<Coef> cf, int l) {
  LinkFlat f;
  const int c = lk[l].cid;
  f.nbr = lk[l].nbr;
  f.u = cf[c].u;
  f.iphi = z128{-cf[c].phi.im, cf[c].phi.re};
  f.psi = z128{cf[c].psi.re, cf[c].psi.im};
  f.dir = z128{cf[c].dir.re, cf[c].dir.im};
  return f;
}

// Element base + off of a state-sized buffer.  A kernel whose lanes share the
// base (a block or an item) passes it apart: the address is then a scalar base
// and a 32-bit lane offset, the same offset for every operand.
struct At {
  long long base;
  int off;
  __device__ __forceinline__ At(long long b, int o = 0) : base(b), off(o) {}
};

__device__ __forceinline__ z128 ldz(const void* p, bool lo, At i) {
  if (!lo) return (static_cast<const z128*>(p) + i.base)[i.off];
  const z64 v = (static_cast<const z64*>(p) + i.base)[i.off];
  return z128{static_cast<double>(v.re), static_cast<double>(v.im)};
}

// ldz with a non-temporal load (streamed operands that later loads must not evict)
__device__ __forceinline__ z128 ldz_nt(const void* p, bool lo, At i) {
  typedef double d2v __attribute__((ext_vector_type(2)));
  typedef float f2v __attribute__((ext_vector_type(2)));
  if (!lo) {
    const d2v w = __builtin_nontemporal_load(static_cast<const d2v*>(p) + i.base + i.off);
    return z128{w.x, w.y};
  }
  const f2v w = __builtin_nontemporal_load(static_cast<const f2v*>(p) + i.base + i.off);
  return z128{static_cast<double>(w.x), static_cast<double>(w.y)};
}

__device__ __forceinline__ void stz(void* p, bool lo, At i, z128 v) {
  if (!lo)
    (static_cast<z128*>(p) + i.base)[i.off] = v;
  else
    (static_cast<z64*>(p) + i.base)[i.off] =
        z64{static_cast<float>(v.re), static_cast<float>(v.im)};
}

__device__ __forceinline__ double zabs(z128 a) { return sqrt(a.re * a.re + a.im * a.im); }

// parity select without indexing kernel-argument arrays by a runtime value
// (which would copy the arguments to scratch memory)
template <typename T>
__device__ __forceinline__ T pick(const T (&a)[2], int cur) {
  return cur ? a[1] : a[0];
}

// Per-element epilogue operands, loaded before the operator work so that
// their memory latency overlaps it.  F64: every operand is complex128.
template <int KP>
struct PreT {
  z128 v[KP];
};
using Pre = PreT<kMaxPre>;

template <bool F64, int KP, bool NT = false>
__device__ __forceinline__ void prefetch(PreT<KP>& p, const StageArgs& A, int cur, At gi,
                                         bool ok) {
#pragma unroll
  for (int s = 0; s < KP; ++s) {
    const void* ptr = cur ? A.pre[1][s] : A.pre[0][s];
    if (ok && s < A.npre && ptr != nullptr)
      p.v[s] = NT ? ldz_nt(ptr, F64 ? false : ((A.pre_lo >> s) & 1u), gi)
                  : ldz(ptr, F64 ? false : ((A.pre_lo >> s) & 1u), gi);
    else
      p.v[s] = z128{0.0, 0.0};
  }
}

// Linear combination sum_s c[s]*p[s] + ck*k, accumulated in s order.  Terms
// with a zero coefficient add an exact zero, so the result equals the
// sequential sum over the non-zero terms (reference order).  P1: operand 1 is p1.
template <bool P1, int KP, class C>
__device__ __forceinline__ z128 combine(const PreT<KP>& p, z128 p1, const C& c, int npre,
                                        double ck, z128 k) {
  z128 v{0.0, 0.0};
#pragma unroll
  for (int s = 0; s < KP; ++s) {
    if (s < npre) {
      const z128 q = P1 && s == 1 ? p1 : p.v[s];
      v.re = fma(c[s], q.re, v.re);
      v.im = fma(c[s], q.im, v.im);
    }
  }
  v.re = fma(ck, k.re, v.re);
  v.im = fma(ck, k.im, v.im);
  return v;
}

// k = -alpha * D
__device__ __forceinline__ z128 scaled_k(z128 alpha, z128 D) {
  return z128{-(alpha.re * D.re - alpha.im * D.im), -(alpha.re * D.im + alpha.im * D.re)};
}

// Epilogue shared by all operator kernels.  D is the operator applied to the
// stage input at flat element gi; returns w^2 of the error norm (or 0).
// AHEAD: the coefficients as the compiler schedules them (see below).
template <bool F64, typename R, int KP, Epi E, bool AHEAD = false>
__device__ __forceinline__ double epilogue(const PreT<KP>& p, const StageArgs& A, int cur, At gi,
                                           cx<R> Dr, z128 alpha) {
  const z128 D = conv<double>(Dr);
  const z128 k = scaled_k(alpha, D);
  z128 p1{0.0, 0.0};
  if constexpr (E == EPI_RK) {
    if (A.mode == MODE_DIFF) {
      z128 v = k;
      if (A.npre > 0) {
        const z128 o = p.v[0];
        v = z128{A.b_re * o.re - A.b_im * o.im + k.re, A.b_re * o.im + A.b_im * o.re + k.im};
      }
      stz(pick(A.dst[0], cur), F64 ? false : A.dst_lo[0], gi, v);
      return 0.0;
    }
  } else if constexpr (E == EPI_K) {
    if (void* kp = pick(A.k, cur)) stz(kp, !F64, gi, k);
    // k_1 of the stored derivative, rounded as a stored k_1 would be
    p1 = scaled_k(alpha, p.v[1]);
    if (!F64) p1 = conv<double>(conv<float>(p1));
  } else {
    stz(pick(A.k, cur), !F64, gi, D);
  }
  // The coefficients are read from the kernel's arguments (FormDev, StageArgs) where they
  // are used: read as A.cc, the compiler loads them ahead of the operator work and spills
  // scalar registers across it (20 levels, FP64: RK4 pass 22.4 us, 21.4 here).  With more
  // than four operands that takes a barrier besides (7-site stages 5 and 6: 36 spills, 20.4
  // and 20.8 us; 0 and 19.2 and 19.6 us).
  static_assert(sizeof(FormDev) % alignof(StageArgs) == 0, "second kernel argument");
  auto ca = reinterpret_cast<cptr<StageArgs>>(
      (cptr<char>)__builtin_amdgcn_kernarg_segment_ptr() + sizeof(FormDev));
  if constexpr (E == EPI_K && KP > 4 && !AHEAD) asm volatile("" : "+s"(ca));
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    if (c < A.ncombo) {
      const z128 v = AHEAD ? combine<E == EPI_K>(p, p1, A.cc[c], A.npre, A.ck[c], k)
                           : combine<E == EPI_K>(p, p1, ca->cc[c], A.npre, ca->ck[c], k);
      stz(pick(A.dst[c], cur), F64 ? false : A.dst_lo[c], gi, v);
      if (void* d2 = pick(A.dst2[c], cur)) stz(d2, F64 ? false : A.dst2_lo[c], gi, v);
    }
  }
  if constexpr (E == EPI_D) {
    if (A.do_err) {
      // operands: the error sum of the six stages before, y_new, y_old
      const z128 e{fma(A.ek, k.re, p.v[0].re), fma(A.ek, k.im, p.v[0].im)};
      const double a1 = zabs(p.v[1]), a0 = zabs(p.v[2]);
      const double w = zabs(e) / (A.atol + A.rtol * (a1 > a0 ? a1 : a0));
      return w * w;
    }
  }
  return 0.0;
}

template <int KP>
using KpTag = std::integral_constant<int, KP>;
template <Epi E>
using EpiTag = std::integral_constant<Epi, E>;

// f(KP, epilogue) of a pass: at most KS operands, or (Dormand-Prince stages that store
// k) KW.
template <int KS, int KW, class F>
void with_epilogue(const StageArgs& A, F&& f) {
  const bool wide = A.npre > KS;
  if (A.npre > KW || (wide && A.epi != EPI_K))
    throw HeomError{HEOM_ERR_STATE, "operator pass: more operands than its kernel takes"};
  if (A.epi == EPI_RK)
    f(KpTag<KS>{}, EpiTag<EPI_RK>{});
  else if (A.epi == EPI_D)
    f(KpTag<KS>{}, EpiTag<EPI_D>{});
  else if (!wide)
    f(KpTag<KS>{}, EpiTag<EPI_K>{});
  else
    f(KpTag<KW>{}, EpiTag<EPI_K>{});
}

// Step control of rkdp::solve_adaptive_step (rkdp.h:97-177) for the attempt
// just finished, followed by the prologue of the next attempt.  The
// std::min/std::max argument orders of the reference are kept so that a NaN
// error norm is handled the same way (factor 10 / 0.2).
__device__ inline void dopri_control(Ctrl* c, double err) {
  const double safety = 0.9, expo = -1.0 / 5.0, dt_min = 1e-16;
  c->err = err;
  c->attempts += 1;
  double dt = c->dt;
  double f = pow(err, expo);
  if (err < 1.0) {
    c->t += dt;
    dt *= safety * ((f < 10.0) ? f : 10.0);
    c->cur ^= 1;
    c->accepted += 1;
    c->count = 0;
    if (c->t >= c->t_bound) {
      c->dt = dt;
      c->done = 1;
      return;
    }
  } else {
    dt *= safety * ((0.2 < f) ? f : 0.2);
    if (dt < dt_min) dt = dt_min;
    c->rejected += 1;
  }
  c->count += 1;
  if (c->count > 1000) {
    c->t = c->t_bound;
    c->done = 1;
    c->gave_up = 1;
    c->dt = dt;
    return;
  }
  if (c->t + dt > c->t_bound) dt = c->t_bound - c->t;
  c->dt = dt;
  // a step that is not positive would never reach t_bound: give up instead
  // (unreachable from a positive step, which the rule above keeps positive)
  if (!(dt > 0.0)) {
    c->t = c->t_bound;
    c->done = 1;
    c->gave_up = 1;
  }
}

// Block reduction of the error-norm partial sums: one value per workgroup,
// written without atomics; dopri_step_kernel combines them.
__device__ inline void write_partial(const StageArgs& A, double v) {
  __shared__ double s_red[16];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nw = (blockDim.x + 63) >> 6;
  if (lane == 0) s_red[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < nw; ++w) t += s_red[w];
    A.partials[blockIdx.x] = t;
  }
}
// Kernel prologue: leave early when the control block says the interval is
// done, pick the ping-pong parity and the step.
struct Prologue {
  int cur;
  z128 alpha;
  bool skip;
};

__device__ __forceinline__ Prologue prologue(const StageArgs& A) {
  Prologue p{0, z128{A.a_re, A.a_im}, false};
  if (A.ctrl) {
    if (A.ctrl->done) {
      p.skip = true;
      return p;
    }
    p.cur = A.ctrl->cur;
    if (A.mode == MODE_STAGE) p.alpha = z128{A.ctrl->dt, 0.0};
  }
  return p;
}

// Learned truncation closure: the network's prediction of the tier-(L+1)
// coupling term of a last-tier ADO, added to D before the epilogue.
template <typename R>
__device__ __forceinline__ void add_closure(const FormDev& d, long long gi, cx<R>& D) {
  if (d.clos == nullptr) return;
  const long long a = gi / d.N2;
  const int r = static_cast<int>(a) - d.clos_lo;
  if (r < 0 || r >= d.clos_n) return;
  const int e = static_cast<int>(gi - a * d.N2);
  const float* y = d.clos + static_cast<long long>(r) * 2 * d.N2;
  for (int p = 0; p < d.clos_parts; ++p) {
    D.re += static_cast<R>(y[e]);
    D.im += static_cast<R>(y[d.N2 + e]);
    y += static_cast<long long>(d.clos_n) * 2 * d.N2;
  }
}
// Partial sum of the error norm of one wavefront (no workgroup barrier),
// written to slot `slot`.
__device__ inline void write_partial_wave(const StageArgs& A, double v, int slot) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((threadIdx.x & 63) == 0) A.partials[slot] = v;
}

// LDS written by a wavefront, then read by other lanes of the same wavefront:
// the LDS serves one wavefront's operations in order, so only the compiler
// must keep them in order.
// The scheduling barrier keeps the code on either side apart, as a workgroup
// barrier would (without it the compiler hoists later loads above the LDS
// phase and holds their registers across it).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  __builtin_amdgcn_sched_barrier(0);
}
inline int cap_grid(long long n) {
  if (n < 1) return 1;
  return n < kMaxGrid ? static_cast<int>(n) : kMaxGrid;
}
// dynamic LDS above 64 KB needs the per-kernel limit raised once
template <typename K>
void allow_lds(K kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    HAMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(bytes)));
}

}  // namespace

}  // namespace hamd
