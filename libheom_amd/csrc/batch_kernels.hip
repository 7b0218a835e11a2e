// Operator pass over a batch of independent Hilbert-form hierarchies.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// ---------------------------------------------------------------------------
// batch of Hilbert-form hierarchies (diagonal V, N <= 8): one persistent
// launch advances every member; a 64-lane wavefront takes IPW consecutive
// work items per step (each 64/N^2 ADOs of one member), loading all of them
// before it computes any (IPW is a tile shape the batch autotuner picks)
// ---------------------------------------------------------------------------
// The lane's share of one work item.
template <typename R, int KP>
struct BatchLane {
  BatchInst I;
  int ado, e, i, j;
  bool ok;
  long long gi;
  cx<R> r;
  PreT<KP> pv;
};

// Load phase of work item `it`: the lane's element, its epilogue operands,
// and the item's H and ADO blocks in LDS.
template <typename R, bool F64, int KP>
__device__ __forceinline__ void batch_load(const FormDev& d, const StageArgs& A, const cx<R>* in,
                                           int it, int cur, int lane, cx<R>* s_rho, cx<R>* s_H,
                                           BatchLane<R, KP>& b) {
  using C = cx<R>;
  const auto items = cst(d.items);
  const auto insts = cst(d.inst);
  const bool live = it < d.n_items;
  const int m = live ? items[it].inst : 0, ado0 = live ? items[it].ado : 0;
  BatchInst& I = b.I;
  I.N = insts[m].N;
  I.N2 = insts[m].N2;
  I.n_hrchy = insts[m].n_hrchy;
  I.apw = insts[m].apw;
  I.ado_base = insts[m].ado_base;
  I.h_off = insts[m].h_off;
  I.tab_off = insts[m].tab_off;
  I.dterm_off = insts[m].dterm_off;
  I.real_v = insts[m].real_v;
  I.coef_off = insts[m].coef_off;
  I.elem_base = insts[m].elem_base;
  const int N = I.N, N2 = I.N2;
  const int la = lane / N2;
  b.e = lane - la * N2;
  b.i = b.e / N;
  b.j = b.e - b.i * N;
  b.ado = ado0 + la;
  b.ok = live && la < I.apw && b.ado < I.n_hrchy;
  b.gi = I.elem_base + static_cast<long long>(b.ok ? b.ado : ado0) * N2 + (b.ok ? b.e : 0);
  b.r = in[b.gi];
  prefetch<F64, KP>(b.pv, A, cur, b.gi, b.ok);
  s_H[lane] = lane < N2 ? conv<R>(d.H[I.h_off + lane]) : C{0, 0};
  s_rho[lane] = b.ok ? b.r : C{0, 0};
}

// Compute phase: D of the lane's element and the Runge-Kutta epilogue.
template <typename R, bool F64, int KP>
__device__ __forceinline__ void batch_compute(const FormDev& d, const StageArgs& A,
                                              const cx<R>* in, int cur, int lane, z128 alpha,
                                              const cx<R>* s_rho, const cx<R>* s_H,
                                              const BatchLane<R, KP>& b, double& err_acc) {
  using C = cx<R>;
  if (!b.ok) return;
  const BatchInst& I = b.I;
  const int N = I.N, N2 = I.N2, i = b.i, j = b.j, e = b.e;
  C acc{0, 0};
  const C* bl = s_rho + (lane / N2) * N2;
  // members have N <= 8: unrolled to 8 with an exit (measured faster than the
  // rolled loop in FP64)
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (k >= N) break;
    cmac(acc, s_H[i * N + k], bl[k * N + j]);
    const C t = bl[i * N + k];
    cmac(acc, C{-t.re, -t.im}, s_H[k * N + j]);
  }
  C D = times_i(acc);
  cmac(D, conv<R>(d.gam[I.ado_base + b.ado]) + conv<R>(d.dterm[I.dterm_off + e]), b.r);
  const int l0 = d.link_ptr[I.ado_base + b.ado], l1 = d.link_ptr[I.ado_base + b.ado + 1];
  // the next link record is loaded with the current link's coefficient,
  // neighbour and table loads (one memory round trip per link instead of two)
  BatchLink qn = l0 < l1 ? d.blink[l0] : BatchLink{0, 0, 0, 0};
  for (int l = l0; l < l1; ++l) {
    const BatchLink ql = qn;
    if (l + 1 < l1) qn = d.blink[l + 1];
    const BatchCoef q = d.bcoef[I.coef_off + ql.cid];
    const C x = in[I.elem_base + static_cast<long long>(ql.nbr) * N2 + e];
    const int tb = ql.u * N2 + e;
    C cf;
    if (I.real_v) {
      const z128 p = d.cmac_tab[I.tab_off + tb];
      cf.re = static_cast<R>(p.re) * static_cast<R>(q.iphi.re) +
              static_cast<R>(p.im) * static_cast<R>(q.psi.re) + static_cast<R>(q.dir.re);
      cf.im = static_cast<R>(p.re) * static_cast<R>(q.iphi.im) +
              static_cast<R>(p.im) * static_cast<R>(q.psi.im) + static_cast<R>(q.dir.im);
    } else {
      cf = conv<R>(d.cmac_tab[I.tab_off + 2 * tb]) * conv<R>(q.iphi) +
           conv<R>(d.cmac_tab[I.tab_off + 2 * tb + 1]) * conv<R>(q.psi) + conv<R>(q.dir);
    }
    cmac(D, cf, x);
  }
  err_acc += epilogue<F64, R, KP>(b.pv, A, cur, b.gi, D, alpha);
}

// KP = 4 for the stages with at most four epilogue operands (every RK4 stage):
// the smaller operand set keeps 7 waves per SIMD (FP32) instead of 4-5.
// WPB wavefronts per workgroup, each with its own items and LDS region and
// none waiting for another (whether that pays is the autotuner's call); the
// error-norm partial sums are one per wavefront.
template <typename R, bool F64, int KP, int IPW, int WPB>
__global__ void __launch_bounds__(64 * WPB) batch_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  __shared__ C s_rho[WPB][IPW][64];
  __shared__ C s_H[WPB][IPW][64];
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int cur = pg.cur;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const int w = WPB > 1 ? __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / 64) : 0;
  const int lane = static_cast<int>(threadIdx.x) - 64 * w;
  double err_acc = 0.0;
  for (int it = (static_cast<int>(blockIdx.x) * WPB + w) * IPW; it < d.n_items;
       it += gridDim.x * WPB * IPW) {
    BatchLane<R, KP> b[IPW];
#pragma unroll
    for (int q = 0; q < IPW; ++q)
      batch_load<R, F64, KP>(d, A, in, it + q, cur, lane, s_rho[w][q], s_H[w][q], b[q]);
    if constexpr (WPB > 1)
      wave_lds_sync();
    else
      __syncthreads();
#pragma unroll
    for (int q = 0; q < IPW; ++q)
      batch_compute<R, F64, KP>(d, A, in, cur, lane, pg.alpha, s_rho[w][q], s_H[w][q], b[q],
                                err_acc);
    if constexpr (WPB > 1)
      wave_lds_sync();
    else
      __syncthreads();
  }
  if (A.do_err) {
    if constexpr (WPB > 1)
      write_partial_wave(A, err_acc, static_cast<int>(blockIdx.x) * WPB + w);
    else
      write_partial(A, err_acc);
  }
}
// rho_S of every batch member, gathered into one block (member order)
__global__ void gather_rho_s_kernel(z128* dst, const z128* src, const BatchInst* inst) {
  const BatchInst I = inst[blockIdx.x];
  for (int e = threadIdx.x; e < I.N2; e += blockDim.x) dst[I.rs_off + e] = src[I.elem_base + e];
}

}  // namespace

template <typename R, bool F64>
int launch_batch(const FormDev& d, const StageArgs& A, hipStream_t st) {
  const int wpb = d.batch_wpb > 0 ? d.batch_wpb : 1;
  // the persistent loop covers every item at any grid; keep one partial slot per wavefront
  const int grid = std::max(1, std::min(d.batch_grid, kMaxGrid / wpb));
  const bool small = A.npre <= 4;
#define HAMD_BATCH(IPW, WPB)                                                               \
{                                                                                        \
  if (small)                                                                             \
    hipLaunchKernelGGL((batch_kernel<R, F64, 4, IPW, WPB>), dim3(grid), dim3(64 * WPB), 0, \
                       st, d, A);                                                        \
  else                                                                                   \
    hipLaunchKernelGGL((batch_kernel<R, F64, kMaxPre, IPW, WPB>), dim3(grid),            \
                       dim3(64 * WPB), 0, st, d, A);                                     \
}
#define HAMD_BATCH_W(IPW)                   \
{                                         \
  if (wpb == 4) HAMD_BATCH(IPW, 4)        \
  else if (wpb == 2) HAMD_BATCH(IPW, 2)   \
  else HAMD_BATCH(IPW, 1)                 \
}
  if (d.batch_ipw == 2) HAMD_BATCH_W(2) else HAMD_BATCH_W(1)
#undef HAMD_BATCH_W
#undef HAMD_BATCH
  return grid * wpb;  // error-norm partials: one per wavefront
}

HAMD_FORM_INSTANCES(launch_batch)

void launch_gather_rho_s(const FormDev& d, void* dst, const void* src, hipStream_t stream) {
  hipLaunchKernelGGL(gather_rho_s_kernel, dim3(d.n_inst), dim3(64), 0, stream,
                     static_cast<z128*>(dst), static_cast<const z128*>(src), d.inst);
  HAMD_HIP(hipGetLastError());
}

}  // namespace hamd
