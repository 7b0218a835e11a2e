// Operator pass over a batch of independent Hilbert-form hierarchies.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// ---------------------------------------------------------------------------
// batch of Hilbert-form hierarchies (diagonal V, N <= 8): one launch advances
// every member; a 64-lane wavefront takes IPW consecutive work items per step
// (each 64/N^2 ADOs of one member), loading all of them before it computes any
// (IPW is a tile shape the batch autotuner picks).
//
// What bounds it: instruction issue first (557 vector instructions per item
// when every lane fetched and converted FP64 tables and divided by a run-time
// N: 75 us of 140 us per stage of a 512-member complex64 sweep, 82 000 items),
// then memory latency and the 64 B (complex64) or 80 B an element of a stage
// must move.  So the tables are stored in the
// operator precision, N = 8, 4 and 2 are compiled in, and a member with one
// ADO per wavefront (N >= 6) reads its links and coefficients as scalars, four
// neighbour loads in flight; smaller members keep per-lane links.  Measured per
// RK4 stage of that sweep (5.0 M elements): complex64 140 -> 82 us (322 MB: 3.9
// TB/s), FP64 145 -> 115 us (400 MB, past the Infinity Cache: 3.5 TB/s).
// ---------------------------------------------------------------------------
constexpr int kBatchPre = 2;  // operands of the fixed-step stages

// The lane's share of one work item.
template <typename R, int KP>
struct BatchLane {
  BatchItem I;
  int e, i, j, la, off;  // off: the element's offset from I.elem
  bool ok;
  cx<R> r, p0, p1;  // rho element, (v_i - v_j, v_i + v_j) of noise 0
  PreT<KP> pv;
};

// V pair of noise row u at element e: real V (v_i - v_j, v_i + v_j) as one
// complex value in p0, complex V as p0 and p1
template <typename R>
__device__ __forceinline__ void batch_vpair(const FormDev& d, const BatchItem& I, int u, int e,
                                            cx<R>& p0, cx<R>& p1) {
  const cx<R>* tab = static_cast<const cx<R>*>(d.b_tab) + I.tab_off;
  const int x = u * I.N * I.N + e;
  if (I.flags & kItemRealV) {
    p0 = tab[x];
  } else {
    p0 = tab[2 * x];
    p1 = tab[2 * x + 1];
  }
}

// Load phase of work item `it`: the lane's element, its epilogue operands,
// and the item's H and ADO blocks in LDS.
template <typename R, bool F64, int KP>
__device__ __forceinline__ void batch_load(const FormDev& d, const StageArgs& A, const cx<R>* in,
                                           int it, int cur, int lane, cx<R>* s_rho, cx<R>* s_H,
                                           BatchLane<R, KP>& b) {
  using C = cx<R>;
  const bool live = it < d.n_items;
  const auto rec = cst(d.items) + (live ? it : 0);
  BatchItem& I = b.I;
  I.elem = rec->elem;
  I.base = rec->base;
  I.N = rec->N;
  I.n_ado = live ? rec->n_ado : 0;
  I.g = rec->g;
  I.l0 = rec->l0;
  I.l1 = rec->l1;
  I.h_off = rec->h_off;
  I.tab_off = rec->tab_off;
  I.dterm_off = rec->dterm_off;
  I.coef_off = rec->coef_off;
  I.flags = rec->flags;
  const int N = I.N, N2 = N * N;
  int la, e, i;
  if (N == 8) {
    la = 0;
    e = lane;
    i = lane >> 3;
  } else if (N == 4) {
    la = lane >> 4;
    e = lane & 15;
    i = e >> 2;
  } else if (N == 2) {
    la = lane >> 2;
    e = lane & 3;
    i = e >> 1;
  } else {
    la = lane / N2;
    e = lane - la * N2;
    i = e / N;
  }
  // lanes without an ADO repeat element 0 of the item and store nothing
  b.ok = la < I.n_ado;
  b.la = b.ok ? la : 0;
  b.e = b.ok ? e : 0;
  b.i = b.ok ? i : 0;
  b.j = b.e - b.i * N;
  b.off = b.la * N2 + b.e;
  b.r = (in + I.elem)[b.off];
  prefetch<F64 || KP == kBatchPre, KP>(b.pv, A, cur, At(I.elem, b.off), true);
  b.p0 = b.p1 = C{0, 0};
  if (I.flags & kItemOneNoise) batch_vpair<R>(d, I, 0, b.e, b.p0, b.p1);
  s_H[lane] = lane < N2 ? static_cast<const C*>(d.b_H)[I.h_off + lane] : C{0, 0};
  s_rho[lane] = b.r;
}

// Compute phase: D of the lane's element.  NS: the member's N (0: any);
// FAST: real V, one noise, no direct links (otherwise read from the item).
template <int NS, bool FAST, typename R, int KP>
__device__ __forceinline__ cx<R> batch_compute(const FormDev& d, const cx<R>* in,
                                               const cx<R>* s_rho, const cx<R>* s_H,
                                               BatchLane<R, KP>& b) {
  using C = cx<R>;
  const BatchItem& I = b.I;
  const int N = NS ? NS : I.N, N2 = N * N, i = b.i, j = b.j, e = b.e;
  C acc{0, 0};
  const C* bl = s_rho + b.la * N2;
  // FP64: two steps at a time (fully unrolled the compiler loads every operand
  // first: 106 instead of 90 VGPRs, 123 instead of 115 us per sweep stage)
  constexpr int KU = sizeof(R) == 8 ? 2 : 8;
#pragma unroll KU
  for (int k = 0; k < (NS ? NS : 8); ++k) {
    if (NS == 0 && k >= N) break;
    cmac(acc, s_H[i * N + k], bl[k * N + j]);
    const C t = bl[i * N + k];
    cmac(acc, C{-t.re, -t.im}, s_H[k * N + j]);
  }
  C D = times_i(acc);
  const bool one = FAST || (I.flags & kItemOneNoise), real = FAST || (I.flags & kItemRealV);
  auto apply = [&](cx<R> iphi, cx<R> psi, cx<R> dir, int u, C x) {
    // with several noises the pair of the link's noise (a zero row for direct links)
    if (!one) batch_vpair<R>(d, I, u, e, b.p0, b.p1);
    C cf;
    if (real) {
      cf.re = b.p0.re * iphi.re + b.p0.im * psi.re + dir.re;
      cf.im = b.p0.re * iphi.im + b.p0.im * psi.im + dir.im;
    } else {
      cf = b.p0 * iphi + b.p1 * psi + dir;
    }
    cmac(D, cf, x);
  };
  const C* nb = in + I.base;
  const C dterm = (static_cast<const C*>(d.b_dterm) + I.dterm_off)[e];
  if (NS ? NS >= 6 : N >= 6) {
    // one ADO per wavefront: uniform links and coefficients
    const auto gp = cst(static_cast<const C*>(d.b_gam)) + I.g;
    cmac(D, C{gp->re, gp->im} + dterm, b.r);
    const auto lks = cst(d.blink);
    const auto cfs = cst(static_cast<const BatchCoef<R>*>(d.b_coef)) + I.coef_off;
    for (int l = I.l0; l < I.l1; l += 4) {
      C x[4];
      int cid[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (l + t < I.l1) {
          cid[t] = lks[l + t].cid;
          x[t] = (nb + static_cast<long long>(lks[l + t].nbr) * N2)[e];
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (l + t < I.l1) {
          const auto q = cfs + cid[t];
          apply(C{q->iphi.re, q->iphi.im}, C{q->psi.re, q->psi.im}, C{q->dir.re, q->dir.im}, q->u,
                x[t]);
        }
      }
    }
  } else {
    const int ado = I.g + b.la;
    cmac(D, static_cast<const C*>(d.b_gam)[ado] + dterm, b.r);
    const BatchCoef<R>* cfs = static_cast<const BatchCoef<R>*>(d.b_coef) + I.coef_off;
    const int l0 = d.link_ptr[ado], l1 = b.ok ? d.link_ptr[ado + 1] : l0;
    // the next link record is loaded with the current link's coefficient and
    // neighbour (one memory round trip per link instead of two)
    Link qn = l0 < l1 ? d.blink[l0] : Link{0, 0};
    for (int l = l0; l < l1; ++l) {
      const Link ql = qn;
      if (l + 1 < l1) qn = d.blink[l + 1];
      const BatchCoef<R> q = cfs[ql.cid];
      const C x = nb[static_cast<long long>(ql.nbr) * N2 + e];
      apply(q.iphi, q.psi, q.dir, q.u, x);
    }
  }
  return D;
}

// KP = 2 for the stages with at most two operands, all complex128 (every RK4
// and lsrk4 stage).
// WPB wavefronts per workgroup, each with its own items and LDS region and
// none waiting for another (whether that pays is the autotuner's call); the
// error-norm partial sums are one per wavefront.
// LOOP: a persistent grid (fewer workgroups than item groups).  With one group
// per workgroup the loop is compiled out: around a loop the compiler keeps every
// kernel argument in scalar registers and spills them (400 lane reads per item).
template <typename R, bool F64, int KP, Epi E, int IPW, int WPB, bool LOOP>
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
  // step g = blockIdx.x, blockIdx.x + gridDim.x, ... runs on XCD g mod 8 (for
  // grids that are multiples of eight) and takes the item group (g mod 8) * per +
  // g / 8: XCD x works through one consecutive eighth of the items, so the
  // neighbour reads of a member meet in one L2 (fetched bytes per stage of the
  // 512-member sweep 1.9x fewer than with items dealt in order)
  const int per = (d.n_items + 8 * WPB * IPW - 1) / (8 * WPB * IPW);
  int g = static_cast<int>(blockIdx.x);
  do {
    const int it = (((g & 7) * per + (g >> 3)) * WPB + w) * IPW;
    BatchLane<R, KP> b[IPW];
#pragma unroll
    for (int q = 0; q < IPW; ++q)
      batch_load<R, F64, KP>(d, A, in, it + q, cur, lane, s_rho[w][q], s_H[w][q], b[q]);
    if constexpr (WPB > 1)
      wave_lds_sync();
    else
      __syncthreads();
#pragma unroll
    for (int q = 0; q < IPW; ++q) {
      C D;
      const bool fast = (b[q].I.flags & kItemFast) == kItemFast;
      if (fast && b[q].I.N == 8)
        D = batch_compute<8, true>(d, in, s_rho[w][q], s_H[w][q], b[q]);
      else if (fast && b[q].I.N == 4)
        D = batch_compute<4, true>(d, in, s_rho[w][q], s_H[w][q], b[q]);
      else if (fast && b[q].I.N == 2)
        D = batch_compute<2, true>(d, in, s_rho[w][q], s_H[w][q], b[q]);
      else
        D = batch_compute<0, false>(d, in, s_rho[w][q], s_H[w][q], b[q]);
      if (b[q].ok)
        err_acc += epilogue<F64, R, KP, E>(b[q].pv, A, cur, At(b[q].I.elem, b[q].off), D, pg.alpha);
    }
    if constexpr (LOOP) {
      if constexpr (WPB > 1)
        wave_lds_sync();
      else
        __syncthreads();
      g += gridDim.x;
    }
  } while (LOOP && g < 8 * per);
  if constexpr (E == EPI_D) {
    if (A.do_err) {
      if constexpr (WPB > 1)
        write_partial_wave(A, err_acc, static_cast<int>(blockIdx.x) * WPB + w);
      else
        write_partial(A, err_acc);
    }
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
  const int ipw = d.batch_ipw == 2 ? 2 : 1;
  const int groups = 8 * ((d.n_items + 8 * wpb * ipw - 1) / (8 * wpb * ipw));
  const int grid = std::max(1, std::min({d.batch_grid, groups, kMaxGrid / wpb}));
  const auto run = [&](auto kp, auto epi) {
    constexpr int KP = decltype(kp)::value;
    constexpr Epi E = decltype(epi)::value;
#define HAMD_BATCH(IPW, WPB)                                                                   \
  {                                                                                            \
    if (grid < groups)                                                                         \
      hipLaunchKernelGGL((batch_kernel<R, F64, KP, E, IPW, WPB, true>), dim3(grid),           \
                         dim3(64 * WPB), 0, st, d, A);                                         \
    else                                                                                       \
      hipLaunchKernelGGL((batch_kernel<R, F64, KP, E, IPW, WPB, false>), dim3(groups),        \
                         dim3(64 * WPB), 0, st, d, A);                                         \
  }
#define HAMD_BATCH_W(IPW)                \
  {                                      \
    if (wpb == 4) HAMD_BATCH(IPW, 4)     \
    else if (wpb == 2) HAMD_BATCH(IPW, 2) \
    else HAMD_BATCH(IPW, 1)              \
  }
    if (ipw == 2) HAMD_BATCH_W(2) else HAMD_BATCH_W(1)
#undef HAMD_BATCH_W
#undef HAMD_BATCH
  };
  if (A.npre <= kBatchPre && A.pre_lo == 0 && A.epi != EPI_D) {
    if (A.epi == EPI_RK)
      run(KpTag<kBatchPre>{}, EpiTag<EPI_RK>{});
    else
      run(KpTag<kBatchPre>{}, EpiTag<EPI_K>{});
  } else if (A.epi == EPI_K) {
    run(KpTag<kMaxPre>{}, EpiTag<EPI_K>{});
  } else if (A.epi == EPI_D) {
    run(KpTag<4>{}, EpiTag<EPI_D>{});  // three operands at most
  } else if constexpr (!F64) {  // a derivative added to a complex64 one
    run(KpTag<kMaxPre>{}, EpiTag<EPI_RK>{});
  } else {
    throw HeomError{HEOM_ERR_STATE, "batch: operands of the pass"};
  }
  return grid * wpb;  // error-norm partials: one per wavefront
}

HAMD_FORM_INSTANCES(launch_batch)

void launch_gather_rho_s(const FormDev& d, void* dst, const void* src, hipStream_t stream) {
  hipLaunchKernelGGL(gather_rho_s_kernel, dim3(d.n_inst), dim3(64), 0, stream,
                     static_cast<z128*>(dst), static_cast<const z128*>(src), d.inst);
  HAMD_HIP(hipGetLastError());
}

}  // namespace hamd
