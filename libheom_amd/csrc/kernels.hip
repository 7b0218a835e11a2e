// HIP kernels of the libheom_amd engine (gfx950).
//
// One kernel pass = one HEOM derivative evaluation fused with the Runge-Kutta
// stage work that consumes it:
//   D_n   = the HEOM operator of heom_hilb.h:108-209 (or its Liouville /
//           global-sparse forms, heom_liou.h:151-255, heom_ado.h:191-202)
//   k     = -dt*D  (calc_diff_impl with alpha = dt, beta = 0; rk4.h:48)
//   y_i+1 = y + sum_j a_ij k_j  (the next stage input, written in the same pass)
//   e     = sum_j E_j k_j and per-workgroup partial sums of the error norm
//           (rkdp.h:142-153); dopri_step_kernel reduces them in a fixed
//           order and runs the step control on the device (rkdp.h:97-177).
//
// Threads map to matrix elements: thread e of an ADO's lane group handles
// element e = i*N + j, so every ADO block (row-major N x N, the reference
// layout) is read and written by contiguous lanes.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// Move the control block on to the next output interval of positive length
// (an interval of no length takes no attempt and keeps the step size); done
// stays set after the last one.
__device__ void next_interval(Ctrl& c, const StepArgs& A) {
  while (c.i_int < A.n_int) {
    const int i = ++c.i_int;
    if (i >= A.n_int) return;
    const double t0 = A.t_list[i], t1 = A.t_list[i + 1];
    if (!(t1 > t0)) continue;
    c.t = t0;
    c.t_bound = t1;
    c.done = 0;
    c.count = 1;
    if (t0 + c.dt > t1) c.dt = t1 - t0;
    return;
  }
}

// The pass between two Dormand-Prince attempts (see StepArgs).  Every workgroup
// sums the partials in the same fixed order and takes the step decision for
// itself (no launch of its own for the decision, no exchange between the
// workgroups); workgroup 0 writes the control block, rho_S at output times
// and the host's progress word.  Then a stream over the state: y and D read, the
// stage input written.  Bound: latency of the reduction (12 650 partials: 101 KB
// per workgroup from L2), then memory.
// The next stage input of an element: y + a21 k, k = -dt D.
template <typename T>
__device__ __forceinline__ void step_input(const StepArgs& A, const z128* y, const T* D, T* sa,
                                           double dt) {
  const z128 alpha{dt, 0.0};
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long x = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; x < A.n;
       x += stride) {
    const z128 k = scaled_k(alpha, conv<double>(D[x])), y0 = y[x];
    z128 v{fma(1.0, y0.re, 0.0), fma(1.0, y0.im, 0.0)};
    v.re = fma(A.a21, k.re, v.re);
    v.im = fma(A.a21, k.im, v.im);
    sa[x] = T{static_cast<decltype(T::re)>(v.re), static_cast<decltype(T::re)>(v.im)};
  }
}

constexpr int kStepBS = 1024;
constexpr int kStepFusedParts = 16384;

__global__ void __launch_bounds__(kStepBS) dopri_step_kernel(const StepArgs A) {
  __shared__ double s_red[kStepBS / 64];
  __shared__ Ctrl s_c;
  __shared__ int s_out[2];  // output times to write: [0] .. [1] - 1
  const bool decide = (A.mode & STEP_CONTROL) && !(A.mode & STEP_FIRST) && !A.prev->done;
  if (decide) {
    double x0 = 0.0, x1 = 0.0, x2 = 0.0, x3 = 0.0;
    int b = threadIdx.x;
    for (; b + 3 * kStepBS < A.nparts; b += 4 * kStepBS) {
      x0 += A.partials[b];
      x1 += A.partials[b + kStepBS];
      x2 += A.partials[b + 2 * kStepBS];
      x3 += A.partials[b + 3 * kStepBS];
    }
    for (; b < A.nparts; b += kStepBS) x0 += A.partials[b];
    double x = (x0 + x1) + (x2 + x3);
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = x;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    Ctrl c = *A.prev;
    s_out[0] = s_out[1] = 0;
    if (decide) {
      double t = 0.0;
      for (int w = 0; w < kStepBS / 64; ++w) t += s_red[w];
      dopri_control(&c, sqrt(t * A.inv_n));
      if (c.done && A.t_list) {
        s_out[0] = c.i_int + 1;
        next_interval(c, A);
        s_out[1] = (c.i_int < A.n_int ? c.i_int : A.n_int) + 1;
      }
    } else if ((A.mode & STEP_FIRST) && A.t_list) {
      s_out[1] = c.i_int + 1;
    }
    if (A.mode & STEP_CONTROL) {
      c.seq += 1;
      if (blockIdx.x == 0) {
        *A.next = c;
        if (A.mail) {
          const bool last =
              !c.done && !(c.t + c.dt < c.t_bound) && (!A.t_list || c.i_int + 1 >= A.n_int);
          __hip_atomic_store(A.mail,
                             static_cast<unsigned long long>(c.seq) << 2 | (last ? 2u : 0u) |
                                 (c.done ? 1u : 0u),
                             __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
      }
    }
    s_c = c;
  }
  __syncthreads();
  const int cur = s_c.cur;
  const z128* y = pick(A.y, cur);
  if (blockIdx.x == 0 && A.rho_s)
    for (int o = s_out[0]; o < s_out[1]; ++o)
      for (int x = threadIdx.x; x < A.n_rs; x += kStepBS)
        A.rho_s[static_cast<long long>(o) * A.n_rs + x] = y[x];
  if (s_c.done || !(A.mode & STEP_INPUT)) return;
  const void* D = pick(A.D, cur);
  if (A.lo)
    step_input(A, y, static_cast<const z64*>(D), static_cast<z64*>(A.sa), s_c.dt);
  else
    step_input(A, y, static_cast<const z128*>(D), static_cast<z128*>(A.sa), s_c.dt);
}
// rho_0 renormalisation (optional): Tr rho_0 of the initial state, then after
// every step rho_0 <- (rho_0 + rho_0^+)/2 * tr0 / Tr, in FP64.  One workgroup of
// 1024 lanes, up to four elements each (n_level <= 64); every element and its
// transpose are read before any lane writes.  y0/y1 (and the FP32 copies f0/f1,
// may be null) are the two parities of the state; ctrl == null: parity 0.
__global__ void __launch_bounds__(1024) rho0_trace_kernel(const z128* y, int N, double* tr0) {
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int i = 0; i < N; ++i) t += y[i * N + i].re;
    *tr0 = t;
  }
}

__global__ void __launch_bounds__(1024) rho0_renorm_kernel(z128* y0, z128* y1, z64* f0, z64* f1,
                                                          Ctrl* ctrl, int N,
                                                          const double* tr0) {
  __shared__ double s_factor;
  // with a control block: project once after each accepted attempt, never after
  // a rejected one or a no-op attempt of a finished interval
  if (ctrl && ctrl->accepted == ctrl->projected) return;
  const int cur = ctrl ? ctrl->cur : 0;
  z128* y = cur ? y1 : y0;
  z64* f = cur ? f1 : f0;
  const int N2 = N * N;
  z128 v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int e = threadIdx.x + r * 1024;
    if (e < N2) {
      const int i = e / N, j = e - i * N;
      const z128 a = y[e], b = y[j * N + i];
      v[r] = z128{0.5 * (a.re + b.re), 0.5 * (a.im - b.im)};
    }
  }
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int i = 0; i < N; ++i) t += y[i * N + i].re;
    const double target = *tr0;
    s_factor = (t != 0.0 && isfinite(t) && isfinite(target)) ? target / t : 1.0;
  }
  __syncthreads();
  const double g = s_factor;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int e = threadIdx.x + r * 1024;
    if (e < N2) {
      const z128 w{g * v[r].re, g * v[r].im};
      y[e] = w;
      if (f) f[e] = z64{static_cast<float>(w.re), static_cast<float>(w.im)};
    }
  }
  if (ctrl && threadIdx.x == 0) ctrl->projected = ctrl->accepted;
}
__global__ void ctrl_init_kernel(Ctrl* c, double t0, double t_bound, double dt, int i_int) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  if (dt < 0.0)
    dt = c->dt;  // keep dt_save (adaptive_step_size_solver.h:39-41,55)
  else
    *c = Ctrl{};  // the start of a solve
  c->t = t0;
  c->t_bound = t_bound;
  c->done = 0;
  c->count = 1;
  c->gave_up = 0;
  c->seq = 0;
  c->i_int = i_int;
  if (t0 + dt > t_bound) dt = t_bound - t0;
  c->dt = dt;
}

__global__ void narrow_kernel(z64* dst, const z128* src, long long n) {
  for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<long long>(gridDim.x) * blockDim.x)
    dst[i] = z64{static_cast<float>(src[i].re), static_cast<float>(src[i].im)};
}

template <typename T>
__global__ void copy_kernel(T* dst, const T* src, long long n) {
  for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<long long>(gridDim.x) * blockDim.x)
    dst[i] = src[i];
}

template <typename R, bool F64>
int launch_form(const FormDev& d, const StageArgs& A, hipStream_t st) {
  switch (d.kind) {
    case HEOM_HILB:
      return launch_hilb<R, F64>(d, A, st);
    case kBatch:
      return launch_batch<R, F64>(d, A, st);
    default:
      return launch_redfield<R, F64>(d, A, st);
  }
}

}  // namespace

int launch_operator(const FormDev& d, int real_bytes, const StageArgs& A, hipStream_t stream) {
  // every operand complex128: the epilogue needs no per-operand type checks
  bool all64 = real_bytes == 8 && !A.in_lo && A.pre_lo == 0 && !A.k_lo;
  for (int c = 0; c < 2; ++c) all64 = all64 && !A.dst_lo[c] && !A.dst2_lo[c];
  int g;
  if (real_bytes == 4)
    g = launch_form<float, false>(d, A, stream);
  else if (all64)
    g = launch_form<double, true>(d, A, stream);
  else  // an FP64 operator never has FP32 operands (Qme::lo)
    throw HeomError{HEOM_ERR_STATE, "operator pass: FP32 operands of an FP64 operator"};
  HAMD_HIP(hipGetLastError());
  return g;
}

// One launch, or, where every workgroup reading every partial would cost more
// than a launch (4.6 us), the decision by one workgroup and then the stage input.
void launch_dopri_step(const StepArgs& A, hipStream_t stream) {
  const long long per = 2 * kStepBS;  // elements per workgroup until the grid is full
  const int grid = static_cast<int>(std::max(1LL, std::min(512LL, (A.n + per - 1) / per)));
  StepArgs a = A;
  if ((a.mode & STEP_CONTROL) && ((a.mode & STEP_INPUT) == 0 || a.nparts > kStepFusedParts)) {
    a.mode &= ~STEP_INPUT;
    hipLaunchKernelGGL(dopri_step_kernel, dim3(1), dim3(kStepBS), 0, stream, a);
    HAMD_HIP(hipGetLastError());
    if (!(A.mode & STEP_INPUT)) return;
    a.mode = STEP_INPUT;
    a.prev = a.next;
    a.rho_s = nullptr;
  }
  hipLaunchKernelGGL(dopri_step_kernel, dim3(grid), dim3(kStepBS), 0, stream, a);
  HAMD_HIP(hipGetLastError());
}

void launch_ctrl_init(Ctrl* c, double t0, double t_bound, double dt, int i_int,
                      hipStream_t stream) {
  hipLaunchKernelGGL(ctrl_init_kernel, dim3(1), dim3(64), 0, stream, c, t0, t_bound, dt, i_int);
  HAMD_HIP(hipGetLastError());
}
void launch_rho0_trace(const void* y, int N, double* tr0, hipStream_t stream) {
  hipLaunchKernelGGL(rho0_trace_kernel, dim3(1), dim3(64), 0, stream, static_cast<const z128*>(y),
                     N, tr0);
  HAMD_HIP(hipGetLastError());
}

void launch_rho0_renorm(void* y0, void* y1, void* f0, void* f1, Ctrl* ctrl, int N,
                        const double* tr0, hipStream_t stream) {
  if (N > 64) throw HeomError{HEOM_ERR_UNSUPPORTED, "renorm_rho0: n_level > 64"};
  hipLaunchKernelGGL(rho0_renorm_kernel, dim3(1), dim3(1024), 0, stream, static_cast<z128*>(y0),
                     static_cast<z128*>(y1), static_cast<z64*>(f0), static_cast<z64*>(f1), ctrl,
                     N, tr0);
  HAMD_HIP(hipGetLastError());
}
void launch_narrow(void* dst, const void* src, long long n, hipStream_t stream) {
  hipLaunchKernelGGL(narrow_kernel, dim3(cap_grid((n + 255) / 256)), dim3(256), 0, stream,
                     static_cast<z64*>(dst), static_cast<const z128*>(src), n);
  HAMD_HIP(hipGetLastError());
}

void launch_copy_grid(void* dst, const void* src, long long n, int grid, hipStream_t stream) {
  hipLaunchKernelGGL((copy_kernel<z128>), dim3(grid), dim3(256), 0, stream, static_cast<z128*>(dst),
                     static_cast<const z128*>(src), n);
  HAMD_HIP(hipGetLastError());
}

void launch_copy(void* dst, const void* src, long long n, int type, hipStream_t stream) {
  const int grid = cap_grid((n + 255) / 256);
  if (type == ST_C128)
    hipLaunchKernelGGL((copy_kernel<z128>), dim3(grid), dim3(256), 0, stream,
                       static_cast<z128*>(dst), static_cast<const z128*>(src), n);
  else
    hipLaunchKernelGGL((copy_kernel<z64>), dim3(grid), dim3(256), 0, stream,
                       static_cast<z64*>(dst), static_cast<const z64*>(src), n);
  HAMD_HIP(hipGetLastError());
}

}  // namespace hamd
