// heom_hilb on the matrix cores (16 < N <= 64), diagonal and dense V.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// ---------------------------------------------------------------------------
// heom_hilb, 16 < N <= 64, diagonal V: the commutator H*rho - rho*H on the
// matrix cores (heom_hilb.h:108-125 computes it with two gemm calls per ADO).
// One ADO per 256-thread workgroup.  rho_n is staged in LDS as separate real
// and imaginary planes with row stride N+1, so that the 16 rows of an MFMA
// fragment fall in distinct banks.  H (shared by every ADO) is read from L2
// as MFMA operands.  Wave w owns NB*NB/4 of the
// (N/16)^2 output tiles, all in one 16-row band, and accumulates H*rho and
// -rho*H into the same accumulators: 4 real products per k step when H is
// real, 8 otherwise.  The accumulators then feed the element-wise part of
// the operator and the fused Runge-Kutta epilogue.
//
// MFMA 16x16xK lane layout (checked against host products): lane l holds
// A[l%16][k0 + l/16] and B[k0 + l/16][l%16] (K = 4), or the 8 consecutive k
// from k0 + 8*(l/16) (bf16, K = 32); accumulator element r of lane l is
// C[4*(l/16) + r][l%16] for the f32 accumulators and C[l/16 + 4*r][l%16]
// for f64.
// ---------------------------------------------------------------------------
typedef double mf_d4 __attribute__((ext_vector_type(4)));
typedef __bf16 mf_b8 __attribute__((ext_vector_type(8)));

template <typename R>
struct Mfma;
template <>
struct Mfma<double> {
  using acc = mf_d4;
  static __device__ __forceinline__ acc mac(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ constexpr int row(int lk, int r) { return lk + 4 * r; }
  static __device__ __forceinline__ const double* re(const FormDev& d) { return d.Hre; }
  static __device__ __forceinline__ const double* im(const FormDev& d) { return d.Him; }
};
template <>
struct Mfma<float> {
  using acc = mf_f4;
  static __device__ __forceinline__ acc mac(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ constexpr int row(int lk, int r) { return 4 * lk + r; }
  static __device__ __forceinline__ const float* re(const FormDev& d) { return d.Hre32; }
  static __device__ __forceinline__ const float* im(const FormDev& d) { return d.Him32; }
};

// x = hi + lo with hi = bf16(x) and lo = bf16(x - hi): 16 significant bits
struct Split8 {
  mf_b8 hi, lo;
};

__device__ __forceinline__ Split8 split8(const float (&x)[8], bool neg) {
  Split8 s;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float v = neg ? -x[q] : x[q];
    const __bf16 h = static_cast<__bf16>(v);
    s.hi[q] = h;
    s.lo[q] = static_cast<__bf16>(v - static_cast<float>(h));
  }
  return s;
}

// a*b ~ hi*hi + hi*lo + lo*hi (the lo*lo term, 2^-16 relative, is dropped);
// the small terms are accumulated first
__device__ __forceinline__ mf_f4 mac3(const Split8& a, const Split8& b, mf_f4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.lo, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, b.hi, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.hi, c, 0, 0, 0);
}

// Coefficient of a neighbour element at (i, j) with the diagonals of every V_u
// in LDS (sv: n_noise + 1 rows of n, the last row zero; real V as R, complex V
// as cx<R>): (v_i - v_j)*iphi + (v_i + v_j)*psi + dir.
template <typename R>
__device__ __forceinline__ cx<R> link_coef_lds(const FormDev& d, const LinkFlat& q, const R* sv,
                                               int n, int i, int j) {
  cx<R> cf;
  if (d.real_v) {
    const R vi = sv[q.u * n + i], vj = sv[q.u * n + j];
    const R c0 = vi - vj, a0 = vi + vj;
    cf.re = c0 * static_cast<R>(q.iphi.re) + a0 * static_cast<R>(q.psi.re) +
            static_cast<R>(q.dir.re);
    cf.im = c0 * static_cast<R>(q.iphi.im) + a0 * static_cast<R>(q.psi.im) +
            static_cast<R>(q.dir.im);
  } else {
    const cx<R>* sc = reinterpret_cast<const cx<R>*>(sv);
    const cx<R> vi = sc[q.u * n + i], vj = sc[q.u * n + j];
    cf = (vi - vj) * conv<R>(q.iphi) + (vi + vj) * conv<R>(q.psi) + conv<R>(q.dir);
  }
  return cf;
}

template <int N>
struct MfmaCfg {
  static constexpr int N2 = N * N;
  static constexpr int LD = N + 1;                // LDS row stride
  static constexpr int NB = N / 16;               // 16-row bands
  // threads per ADO: N = 64 eight waves with two output tiles each, N = 48 nine
  // and N = 32 four with one
  static constexpr int BS = N == 64 ? 512 : N == 48 ? 576 : 256;
  static constexpr int KS = N / 4;                // k steps of the 16x16x4 products
  static constexpr int KB = N / 32;               // k steps of the bf16 products
  static_assert(N == 32 || N == 48 || N == 64, "MFMA path: tiles of 32, 48 or 64 rows");
};

// H*rho - rho*H for the wave's tiles, operands in the state precision R
template <int N, typename R, bool REALH, int TPW>
__device__ __forceinline__ void mfma_commutator(const FormDev& d, const R* s_re, const R* s_im,
                                                int band, int t0, int lr, int lk,
                                                typename Mfma<R>::acc (&cre)[TPW],
                                                typename Mfma<R>::acc (&cim)[TPW]) {
  using M = Mfma<R>;
  using Cfg = MfmaCfg<N>;
  const R* Hr = M::re(d);
  const R* Hi = M::im(d);
  const int row = band * 16 + lr;
  // fewer tiles per wave go with a smaller register budget (see hilb_mfma_kernel)
  constexpr int KU = TPW > 2 ? Cfg::KS : 4;
#pragma unroll KU
  for (int ks = 0; ks < Cfg::KS; ++ks) {
    const int kk = 4 * ks + lk;
    const R arr = -s_re[row * Cfg::LD + kk], ari = -s_im[row * Cfg::LD + kk];
    const R ahr = Hr[row * N + kk], ahi = REALH ? R(0) : Hi[row * N + kk];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int col = ((t0 + t) % Cfg::NB) * 16 + lr;
      const R brr = s_re[kk * Cfg::LD + col], bri = s_im[kk * Cfg::LD + col];
      const R bhr = Hr[kk * N + col];
      cre[t] = M::mac(ahr, brr, cre[t]);   //  Hr rho_r
      cim[t] = M::mac(ahr, bri, cim[t]);   //  Hr rho_i
      cre[t] = M::mac(arr, bhr, cre[t]);   // -rho_r Hr
      cim[t] = M::mac(ari, bhr, cim[t]);   // -rho_i Hr
      if (!REALH) {
        const R bhi = Hi[kk * N + col];
        cre[t] = M::mac(-ahi, bri, cre[t]);  // -Hi rho_i
        cim[t] = M::mac(ahi, brr, cim[t]);   //  Hi rho_r
        cre[t] = M::mac(-ari, bhi, cre[t]);  //  rho_i Hi
        cim[t] = M::mac(arr, bhi, cim[t]);   // -rho_r Hi
      }
    }
  }
}

// the same products on bf16 matrix cores with split operands (FP32 state)
template <int N, bool REALH, int TPW>
__device__ __forceinline__ void mfma_commutator_bf16x3(const FormDev& d, const float* s_re,
                                                       const float* s_im, int band, int t0,
                                                       int lr, int lk, mf_f4 (&cre)[TPW],
                                                       mf_f4 (&cim)[TPW]) {
  using Cfg = MfmaCfg<N>;
  const float* Hr = d.Hre32;
  const float* Hi = d.Him32;
  const int row = band * 16 + lr;
  for (int kb = 0; kb < Cfg::KB; ++kb) {
    const int k0 = 32 * kb + 8 * lk;
    float x[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = Hr[row * N + k0 + q];
    const Split8 ahr = split8(x, false);
    Split8 ahi{}, nahi{};
    if (!REALH) {
#pragma unroll
      for (int q = 0; q < 8; ++q) x[q] = Hi[row * N + k0 + q];
      ahi = split8(x, false);
      nahi = split8(x, true);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = s_re[row * Cfg::LD + k0 + q];
    const Split8 arr = split8(x, true);   // -rho_r
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = s_im[row * Cfg::LD + k0 + q];
    const Split8 ari = split8(x, true);   // -rho_i
    const Split8 pari = split8(x, false);
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int col = ((t0 + t) % Cfg::NB) * 16 + lr;
#pragma unroll
      for (int q = 0; q < 8; ++q) x[q] = s_re[(k0 + q) * Cfg::LD + col];
      const Split8 brr = split8(x, false);
#pragma unroll
      for (int q = 0; q < 8; ++q) x[q] = s_im[(k0 + q) * Cfg::LD + col];
      const Split8 bri = split8(x, false);
#pragma unroll
      for (int q = 0; q < 8; ++q) x[q] = Hr[(k0 + q) * N + col];
      const Split8 bhr = split8(x, false);
      cre[t] = mac3(ahr, brr, cre[t]);
      cim[t] = mac3(ahr, bri, cim[t]);
      cre[t] = mac3(arr, bhr, cre[t]);
      cim[t] = mac3(ari, bhr, cim[t]);
      if (!REALH) {
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = Hi[(k0 + q) * N + col];
        const Split8 bhi = split8(x, false);
        cre[t] = mac3(nahi, bri, cre[t]);
        cim[t] = mac3(ahi, brr, cim[t]);
        cre[t] = mac3(pari, bhi, cre[t]);
        cim[t] = mac3(arr, bhi, cim[t]);
      }
    }
  }
}

// BS threads (BS / 64 waves) per ADO; every form asks for two workgroups per
// CU (LDS holds two FP64 workgroups per CU), i.e. BS / 128 waves per SIMD:
// 256 threads leave 256 registers per lane, 512 threads 128.
// BF16X3: R = float, products via mfma_commutator_bf16x3.  N is the tile size
// (mfma_tile: 32, 48 or 64); the ADO block is n x n with n = d.N <= N, zero-padded in
// LDS (and H in its planes), so that the padded rows and columns of the products are
// exactly zero.
template <int N, typename R, bool REALH, bool F64, int KP, Epi E, bool BF16X3, bool PADDED,
          int BS>
__global__ void __launch_bounds__(BS, BS / 128)
    hilb_mfma_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  using M = Mfma<R>;
  using Cfg = MfmaCfg<N>;
  constexpr int N2 = Cfg::N2, LD = Cfg::LD, NB = Cfg::NB;
  constexpr int TPW = NB * NB / (BS / 64);  // output tiles per wave
  static_assert(TPW >= 1 && TPW * (BS / 64) == NB * NB, "tiles must divide among the waves");
  extern __shared__ __align__(16) unsigned char s_dyn[];
  R* s_re = reinterpret_cast<R*>(s_dyn);
  R* s_im = s_re + N * LD;
  R* s_v = s_im + N * LD;  // diagonals of every V_u (and a zero row), see link_coef_lds
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  // the ADO block (n <= N); unpadded blocks keep the index arithmetic constant
  const int n = PADDED ? d.N : N, n2 = PADDED ? d.N2 : N * N;
  if (PADDED) {  // the padding stays zero: only rows and columns < n are ever written
    for (int x = threadIdx.x; x < 2 * N * LD; x += BS) s_re[x] = R(0);
  }
  {
    const int nvd = (d.n_noise + 1) * d.N, nvd0 = d.n_noise * d.N;
    for (int x = threadIdx.x; x < nvd; x += BS) {
      const z128 v = x < nvd0 ? d.Vd[x] : z128{0.0, 0.0};
      if (d.real_v) {
        s_v[x] = static_cast<R>(v.re);
      } else {
        s_v[2 * x] = static_cast<R>(v.re);
        s_v[2 * x + 1] = static_cast<R>(v.im);
      }
    }
  }
  __syncthreads();
  const int cur = pg.cur;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const auto link_ptr = cst(d.link_ptr);
  const auto flat = cst(d.flat);
  const auto gam = cst(d.gam);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int t0 = wave * TPW;
  const int band = t0 / NB;
  double err_acc = 0.0;
  for (int w = blockIdx.x; w < d.n_hrchy; w += gridDim.x) {
    // work unit w: the XCD-aware block map when present
    BlockMap bm{w, 0, 0, 0};
    if (d.bmap) {
      const auto p = cst(d.bmap) + w;
      bm = BlockMap{p->g, p->l0, p->l1, 0};
    } else {
      bm.l0 = link_ptr[w];
      bm.l1 = link_ptr[w + 1];
    }
    const int g = bm.g;
    const long long base = static_cast<long long>(g) * n2;
    {
      // all loads of rho_n in flight before the LDS stores
      constexpr int PER = N2 / BS;
      C v[PER];
#pragma unroll
      for (int c = 0; c < PER; ++c) {
        const int x = threadIdx.x + c * BS;
        v[c] = x < n2 ? in[base + x] : C{0, 0};
      }
#pragma unroll
      for (int c = 0; c < PER; ++c) {
        const int x = threadIdx.x + c * BS;
        if (x < n2) {
          const int i = x / n, j = x - (x / n) * n;
          s_re[i * LD + j] = v[c].re;
          s_im[i * LD + j] = v[c].im;
        }
      }
    }
    __syncthreads();
    typename M::acc cre[TPW], cim[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      cre[t] = typename M::acc{0, 0, 0, 0};
      cim[t] = typename M::acc{0, 0, 0, 0};
    }
    if constexpr (BF16X3)
      mfma_commutator_bf16x3<N, REALH, TPW>(d, s_re, s_im, band, t0, lr, lk, cre, cim);
    else
      mfma_commutator<N, R, REALH, TPW>(d, s_re, s_im, band, t0, lr, lk, cre, cim);
    // every wave has read rho_n as MFMA operands: each lane now replaces its
    // own elements by i[H, rho] + (Gamma_n + delta term) rho (one owner each)
    __syncthreads();
    const C gm = conv<R>(z128{gam[g].re, gam[g].im});
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int col = ((t0 + t) % NB) * 16 + lr;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = band * 16 + M::row(lk, r);
        if (i < n && col < n) {
          C D = times_i(C{cre[t][r], cim[t][r]});
          const C rv{s_re[i * LD + col], s_im[i * LD + col]};
          cmac(D, gm + conv<R>(d.dterm[i * n + col]), rv);
          s_re[i * LD + col] = D.re;
          s_im[i * LD + col] = D.im;
        }
      }
    }
    __syncthreads();
    // Neighbour couplings and the Runge-Kutta epilogue, element-parallel and
    // coalesced.  Two schedules of the same per-element arithmetic (D, then
    // the links in order, then the epilogue):
    //  - links outer (FP64 and BF16X3 forms, and every form with eight waves
    //    per ADO): for each link the loads of LCH of the thread's elements of
    //    the neighbour block are in flight together; each thread updates only
    //    its own elements (x = tid + c*BS) in LDS and reads them back in the
    //    epilogue, so the phases need no barrier;
    //  - links inside the epilogue passes (complex64 form with four waves per
    //    ADO, whose register budget keeps three waves per SIMD that way).
    // Each epilogue pass takes CH elements per thread and issues every load
    // before its stores (the stores may alias later loads); elements past the
    // block read element 0 and store nothing.
    constexpr bool kLinksOuter = sizeof(R) == 8 || BF16X3 || BS > 256;
    constexpr int EPT = N2 / BS;              // elements per thread (tile)
    constexpr int LMAX = BS > 256 ? 4 : 8;    // register budget: 256 / 128 per lane
    constexpr int LCH = EPT < LMAX ? EPT : LMAX;  // elements per load group
    constexpr int CH = (KP <= 4 && BS <= 256) ? 2 : 1;
    const int l0 = bm.l0, l1 = bm.l1;
    if constexpr (kLinksOuter) {
      for (int l = l0; l < l1; ++l) {
        const LinkFlat q = ld_flat(flat + l);
        const C* nb = in + static_cast<long long>(q.nbr) * n2;
#pragma unroll 1
        for (int c0 = 0; c0 < EPT; c0 += LCH) {
          C xv[LCH];
#pragma unroll
          for (int c = 0; c < LCH; ++c) {
            const int x = threadIdx.x + (c0 + c) * BS;
            const int xs = x < n2 ? x : 0;
            xv[c] = nb[xs];
          }
#pragma unroll
          for (int c = 0; c < LCH; ++c) {
            const int x = threadIdx.x + (c0 + c) * BS;
            if (x < n2) {
              const int i = x / n, j = x - (x / n) * n;
              C Dv{s_re[i * LD + j], s_im[i * LD + j]};
              cmac(Dv, link_coef_lds<R>(d, q, s_v, d.N, i, j), xv[c]);
              s_re[i * LD + j] = Dv.re;
              s_im[i * LD + j] = Dv.im;
            }
          }
        }
      }
    }
    for (int x0 = threadIdx.x; x0 < n2; x0 += BS * CH) {
      C Dc[CH];
      PreT<KP> pv[CH];
      int xs[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int x = x0 + c * BS;
        xs[c] = x < n2 ? x : 0;
        const int i = xs[c] / n, j = xs[c] - (xs[c] / n) * n;
        Dc[c] = C{s_re[i * LD + j], s_im[i * LD + j]};
        // FP64 at N = 64: the streamed epilogue operands are loaded non-temporally,
        // which keeps more of the stage input (the neighbour blocks) cached
        prefetch<F64, KP, sizeof(R) == 8 && N == 64>(pv[c], A, cur, base + xs[c], true);
      }
      if constexpr (!kLinksOuter) {
        for (int l = l0; l < l1; ++l) {
          const LinkFlat q = ld_flat(flat + l);
          C xv[CH];
#pragma unroll
          for (int c = 0; c < CH; ++c) xv[c] = in[static_cast<long long>(q.nbr) * n2 + xs[c]];
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            const int i = xs[c] / n, j = xs[c] - (xs[c] / n) * n;
            cmac(Dc[c], link_coef_lds<R>(d, q, s_v, d.N, i, j), xv[c]);
          }
        }
      }
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int x = x0 + c * BS;
        if (x < n2) {
          add_closure(d, base + x, Dc[c]);
          // FP64 at N = 64 reads the coefficients ahead of its eight passes: Dormand-Prince
          // pass of 969 ADOs 117.1 us on average, 121.2 read in each pass (RK4 and the
          // other sizes and types are 1-6% faster with the latter)
          err_acc += epilogue<F64, R, KP, E, sizeof(R) == 8 && N == 64 && E == EPI_K>(
              pv[c], A, cur, base + x, Dc[c], pg.alpha);
        }
      }
    }
    __syncthreads();
  }
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, err_acc);
}

// ---------------------------------------------------------------------------
// heom_hilb on matrix cores with dense (non-diagonal) V, 16 < N <= 64
// (heom_hilb.h:108-209): per ADO
//   D = i[H, rho] + Gamma_n rho + sum_u (V_u X_u + Y_u V_u) + sum_direct dir rho_l
//   X_u = i Phi_u + Psi_u + delta_u [V_u, rho],  Y_u = Psi_u - i Phi_u - delta_u [V_u, rho]
// (i[V,Phi] + {V,Psi} + delta [V,[V,rho]] = V X + Y V).  A lane works on the
// elements of its accumulators throughout: D stays in the accumulators from
// i[H, rho] + Gamma rho on; per noise [V_u, rho] goes to a second accumulator set,
// the links of noise u add to X_u and Y_u in registers (one read of each neighbour
// for both), and the two are written to the LDS workspace one after the other as
// operands of the next products.  The epilogue needs no exchange either.
// Bound: the matrix pipe (18 real-operand products of N^3 per ADO with four
// noises), 53% busy at N = 64: one workgroup per CU, phases between barriers.
// 969 ADOs, four noises, FP64 / complex64, us: with X and Y accumulated in LDS by
// separate passes over the links 64 levels 491 / 300, 20 levels 98 / 73; now 437 / 267
// and 74 / 64; with tiles of 48 rows besides, 40 levels 440 / 276 -> 259 / 222.
// ---------------------------------------------------------------------------
constexpr int kCprodAhead = 4;

// acc += sgn * (A B) for the wave's tiles.  A and B are complex; an operand in
// LDS has leading dimension LD, a global one (a V_u plane pair) N, and a global
// operand is real when GREAL (its imaginary plane is not read).  Global operands
// come from L2, 500 cycles and more away, and a SIMD has two or three waves to
// hide that: KG k steps are loaded ahead of their products (two at a time cost
// 3% of the stage at N = 64, eight at a time as much in registers).
template <int N, typename R, bool A_LDS, bool B_LDS, bool GREAL, int TPW>
__device__ __forceinline__ void mfma_cprod(const R* ar, const R* ai, const R* br, const R* bi,
                                           R sgn, int band, int t0, int lr, int lk,
                                           typename Mfma<R>::acc (&cre)[TPW],
                                           typename Mfma<R>::acc (&cim)[TPW]) {
  using M = Mfma<R>;
  using Cfg = MfmaCfg<N>;
  constexpr int LDA = A_LDS ? Cfg::LD : N, LDB = B_LDS ? Cfg::LD : N;
  constexpr bool AR = !A_LDS && GREAL, BR = !B_LDS && GREAL;
  constexpr int KG = GREAL ? kCprodAhead : 2;
  static_assert(Cfg::KS % KG == 0, "k groups");
  const int row = band * 16 + lr;
  R ga_r[KG], ga_i[KG], gb_r[KG][TPW], gb_i[KG][TPW];
  auto load = [&](int k0) {
#pragma unroll
    for (int s = 0; s < KG; ++s) {
      const int kk = 4 * (k0 + s) + lk;
      if (!A_LDS) {
        ga_r[s] = ar[row * LDA + kk];
        if (!AR) ga_i[s] = ai[row * LDA + kk];
      }
      if (!B_LDS) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
          const int col = ((t0 + t) % Cfg::NB) * 16 + lr;
          gb_r[s][t] = br[kk * LDB + col];
          if (!BR) gb_i[s][t] = bi[kk * LDB + col];
        }
      }
    }
  };
#pragma unroll 1
  for (int k0 = 0; k0 < Cfg::KS; k0 += KG) {
    load(k0);
#pragma unroll
    for (int s = 0; s < KG; ++s) {
      const int kk = 4 * (k0 + s) + lk;
      const R a_r = sgn * (A_LDS ? ar[row * LDA + kk] : ga_r[s]);
      const R a_i = AR ? R(0) : sgn * (A_LDS ? ai[row * LDA + kk] : ga_i[s]);
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        const int col = ((t0 + t) % Cfg::NB) * 16 + lr;
        const R b_r = B_LDS ? br[kk * LDB + col] : gb_r[s][t];
        cre[t] = M::mac(a_r, b_r, cre[t]);
        if (!BR) {
          const R b_i = B_LDS ? bi[kk * LDB + col] : gb_i[s][t];
          cim[t] = M::mac(a_r, b_i, cim[t]);
          if (!AR) cre[t] = M::mac(-a_i, b_i, cre[t]);
        }
        if (!AR) cim[t] = M::mac(a_i, b_r, cim[t]);
      }
    }
  }
}

template <typename R>
struct MfmaV;
template <>
struct MfmaV<double> {
  static __device__ __forceinline__ const double* re(const FormDev& d) { return d.Vre; }
  static __device__ __forceinline__ const double* im(const FormDev& d) { return d.Vim; }
};
template <>
struct MfmaV<float> {
  static __device__ __forceinline__ const float* re(const FormDev& d) { return d.Vre32; }
  static __device__ __forceinline__ const float* im(const FormDev& d) { return d.Vim32; }
};

// elements per thread of rho_n whose loads are in flight together
constexpr int kDenseCh = 4;
// waves per SIMD the registers have to allow: one workgroup per CU at N = 64 in FP64
// (133 KB of LDS), two in FP32
template <int N, typename R>
constexpr int kDenseWps = sizeof(R) == 4 ? 4 : N == 64 ? 2 : 3;

template <int N, typename R, bool REALV, bool REALH, bool F64, int KP, Epi E, bool PADDED, int BS>
__global__ void __launch_bounds__(BS, (kDenseWps<N, R>))
    hilb_mfma_dense_kernel(const FormDev d, const StageArgs A) {
  using C = cx<R>;
  using M = Mfma<R>;
  using Cfg = MfmaCfg<N>;
  using acc_t = typename M::acc;
  constexpr int N2 = Cfg::N2, LD = Cfg::LD, NB = Cfg::NB;
  constexpr int TPW = NB * NB / (BS / 64);  // output tiles per wave
  constexpr int EPT = N2 / BS;  // elements per thread when rho_n is staged
  extern __shared__ __align__(16) unsigned char s_dyn[];
  R* s_re = reinterpret_cast<R*>(s_dyn);  // rho_n
  R* s_im = s_re + N * LD;
  R* w_re = s_im + N * LD;  // workspace: X_u, then Y_u
  R* w_im = w_re + N * LD;
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const int n = PADDED ? d.N : N, n2 = PADDED ? d.N2 : N * N;
  if (PADDED) {  // the padding stays zero: only rows and columns < n are ever written
    for (int x = threadIdx.x; x < 4 * N * LD; x += BS) s_re[x] = R(0);
    __syncthreads();
  }
  const int cur = pg.cur;
  const C* in = static_cast<const C*>(pick(A.in, cur));
  const auto link_ptr = cst(d.link_ptr);
  const auto flat = cst(d.flat);
  const auto gam = cst(d.gam);
  const auto sdl = cst(d.sdelta);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int t0 = wave * TPW;
  const int band = t0 / NB;
  const R* Vr0 = MfmaV<R>::re(d);
  const R* Vi0 = MfmaV<R>::im(d);
  // the lane's elements: those of its accumulators, (i0 + r RS, j0 + 16 t), all tiles in
  // one band (padding: element 0, not stored)
  constexpr int RS = M::row(0, 1);
  const int i0 = band * 16 + M::row(lk, 0), j0 = (t0 % NB) * 16 + lr, off0 = i0 * n + j0;
  bool in_block[TPW][4];
  int at[TPW][4];
#pragma unroll
  for (int t = 0; t < TPW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      in_block[t][r] = !PADDED || (i0 + r * RS < n && j0 + 16 * t < n);
      at[t][r] = in_block[t][r] ? off0 + r * RS * n + 16 * t : 0;
    }
  double err_acc = 0.0;
  for (int w = blockIdx.x; w < d.n_hrchy; w += gridDim.x) {
    BlockMap bm{w, 0, 0, 0};
    if (d.bmap) {
      const auto p = cst(d.bmap) + w;
      bm = BlockMap{p->g, p->l0, p->l1, 0};
    } else {
      bm.l0 = link_ptr[w];
      bm.l1 = link_ptr[w + 1];
    }
    const int g = bm.g;
    const long long base = static_cast<long long>(g) * n2;
#pragma unroll 1
    for (int c0 = 0; c0 < EPT; c0 += kDenseCh) {
      C v[kDenseCh];
#pragma unroll
      for (int c = 0; c < kDenseCh; ++c) {
        const int x = threadIdx.x + (c0 + c) * BS;
        v[c] = x < n2 ? in[base + x] : C{0, 0};
      }
#pragma unroll
      for (int c = 0; c < kDenseCh; ++c) {
        const int x = threadIdx.x + (c0 + c) * BS;
        if (x < n2) {
          const int i = x / n, j = x - (x / n) * n;
          s_re[i * LD + j] = v[c].re;
          s_im[i * LD + j] = v[c].im;
        }
      }
    }
    __syncthreads();
    acc_t cre[TPW], cim[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      cre[t] = acc_t{0, 0, 0, 0};
      cim[t] = acc_t{0, 0, 0, 0};
    }
    mfma_commutator<N, R, REALH, TPW>(d, s_re, s_im, band, t0, lr, lk, cre, cim);
    // D = i[H, rho] + Gamma_n rho at the accumulator positions
    const C gm = conv<R>(z128{gam[g].re, gam[g].im});
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int col = ((t0 + t) % NB) * 16 + lr;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = band * 16 + M::row(lk, r);
        const C rv{s_re[i * LD + col], s_im[i * LD + col]};
        C Dv = times_i(C{cre[t][r], cim[t][r]});
        cmac(Dv, gm, rv);
        cre[t][r] = Dv.re;
        cim[t][r] = Dv.im;
      }
    }
    const int nn = d.n_noise;
    int l = bm.l0;
    for (int u = 0; u < nn; ++u) {
      const R* Vr = Vr0 + static_cast<size_t>(u) * N2;
      const R* Vi = Vi0 + static_cast<size_t>(u) * N2;
      acc_t ccr[TPW], cci[TPW];
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        ccr[t] = acc_t{0, 0, 0, 0};
        cci[t] = acc_t{0, 0, 0, 0};
      }
      // C = V rho - rho V
      mfma_cprod<N, R, false, true, REALV, TPW>(Vr, Vi, s_re, s_im, R(1), band, t0, lr, lk, ccr,
                                                cci);
      mfma_cprod<N, R, true, false, REALV, TPW>(s_re, s_im, Vr, Vi, R(-1), band, t0, lr, lk, ccr,
                                                cci);
      const C dl = conv<R>(z128{sdl[u].re, sdl[u].im});
      // links of noise u: [lu0, lu1) (the links of an ADO are sorted by noise)
      const int lu0 = l;
      while (l < bm.l1 && flat[l].u == u) ++l;
      const int lu1 = l;
      // X = delta C + sum (iphi + psi) rho_l and Y = sum (psi - iphi) rho_l - delta C at the
      // accumulator positions: the neighbours are read once for both
      C xs[TPW][4], ys[TPW][4];
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          xs[t][r] = dl * C{ccr[t][r], cci[t][r]};
          ys[t][r] = C{-xs[t][r].re, -xs[t][r].im};
        }
      for (int lq = lu0; lq < lu1; ++lq) {
        const LinkFlat q = ld_flat(flat + lq);
        const C ip = conv<R>(q.iphi), ps = conv<R>(q.psi);
        const C cx = ip + ps, cy = ps - ip;
        const C* nb = in + static_cast<long long>(q.nbr) * n2;
        C xv[TPW][4];
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) xv[t][r] = nb[at[t][r]];
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            cmac(xs[t][r], cx, xv[t][r]);
            cmac(ys[t][r], cy, xv[t][r]);
          }
      }
      auto put = [&](const C (&v)[TPW][4]) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
          const int col = ((t0 + t) % NB) * 16 + lr;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = band * 16 + M::row(lk, r);
            if (in_block[t][r]) {
              w_re[i * LD + col] = v[t][r].re;
              w_im[i * LD + col] = v[t][r].im;
            }
          }
        }
        __syncthreads();
      };
      put(xs);  // D += V X
      mfma_cprod<N, R, false, true, REALV, TPW>(Vr, Vi, w_re, w_im, R(1), band, t0, lr, lk, cre,
                                                cim);
      __syncthreads();
      put(ys);  // D += Y V
      mfma_cprod<N, R, true, false, REALV, TPW>(w_re, w_im, Vr, Vi, R(1), band, t0, lr, lk, cre,
                                                cim);
      __syncthreads();
    }
    // direct links (off-diagonal gamma) and the Runge-Kutta epilogue
    const int ld0 = l;
    C D[TPW][4];
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) D[t][r] = C{cre[t][r], cim[t][r]};
    for (int lq = ld0; lq < bm.l1; ++lq) {
      const LinkFlat q = ld_flat(flat + lq);
      const C dir = conv<R>(q.dir);
      const C* nb = in + static_cast<long long>(q.nbr) * n2;
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) cmac(D[t][r], dir, nb[at[t][r]]);
    }
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        PreT<KP> pv;
        prefetch<F64, KP>(pv, A, cur, base + at[t][r], true);
        if (in_block[t][r]) {
          add_closure(d, base + at[t][r], D[t][r]);
          err_acc += epilogue<F64, R, KP, E>(pv, A, cur, base + at[t][r], D[t][r], pg.alpha);
        }
      }
    __syncthreads();  // every wave has finished reading rho
  }
  if constexpr (E == EPI_D)
    if (A.do_err) write_partial(A, err_acc);
}

template <int N, typename R, bool F64, bool BF16X3>
int launch_hilb_mfma_n(const FormDev& d, const StageArgs& A, hipStream_t st) {
  // rho_n planes, then the diagonals of every V_u and a zero row
  const size_t lds = 2 * sizeof(R) * N * MfmaCfg<N>::LD +
                     sizeof(R) * (d.real_v ? 1 : 2) * static_cast<size_t>(d.n_noise + 1) * d.N;
  if (lds > kMfmaLdsCap)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "matrix-core path: too many noises for LDS"};
  const int grid = cap_grid(d.n_hrchy);
  // N = 64: eight waves per ADO, each with half the output tiles (two
  // workgroups per CU either way, so twice the waves work on the same ADOs;
  // measured at 969 ADOs per Dormand-Prince stage: FP64 135 against 158 us,
  // split-bf16 99 against 138 us, complex64 with the links outer 112 against
  // 126 us)
  constexpr int BS = MfmaCfg<N>::BS;
  const auto run = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(BS), lds, st, d, A);
  };
  with_epilogue<4, kMaxPre>(A, [&](auto kp, auto epi) {
    constexpr int KP = decltype(kp)::value;
    constexpr Epi E = decltype(epi)::value;
#define HAMD_MFMA(REALH, PAD)                                             \
  {                                                                       \
    auto k = hilb_mfma_kernel<N, R, REALH, F64, KP, E, BF16X3, PAD, BS>; \
    static bool once = (allow_lds(k, kMfmaLdsCap), true);                 \
    (void)once;                                                           \
    run(k);                                                               \
  }
    if (d.real_h) {
      if (d.N == N) HAMD_MFMA(true, false) else HAMD_MFMA(true, true)
    } else {
      if (d.N == N) HAMD_MFMA(false, false) else HAMD_MFMA(false, true)
    }
#undef HAMD_MFMA
  });
  return grid;
}

template <int N, typename R, bool F64>
int launch_hilb_mfma_dense_n(const FormDev& d, const StageArgs& A, hipStream_t st) {
  // rho_n planes and the workspace planes
  const size_t lds = 4 * sizeof(R) * N * MfmaCfg<N>::LD;
  if (lds > kMfmaLdsCap)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "matrix-core path: the blocks exceed LDS"};
  const int grid = cap_grid(d.n_hrchy);
  // N = 64: eight waves per ADO (measured at 969 ADOs: 497 against 715 us per
  // FP64 stage, 309 against 364 us complex64)
  constexpr int BS = MfmaCfg<N>::BS;
  const auto run = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(BS), lds, st, d, A);
  };
  with_epilogue<4, kMaxPre>(A, [&](auto kp, auto epi) {
    constexpr int KP = decltype(kp)::value;
    constexpr Epi E = decltype(epi)::value;
#define HAMD_MD(REALV, REALH, PAD)                                             \
  {                                                                            \
    auto k = hilb_mfma_dense_kernel<N, R, REALV, REALH, F64, KP, E, PAD, BS>; \
    static bool once = (allow_lds(k, kMfmaLdsCap), true);                      \
    (void)once;                                                                \
    run(k);                                                                    \
  }
#define HAMD_MD_P(REALV, REALH) \
  {                             \
    if (d.N == N) HAMD_MD(REALV, REALH, false) else HAMD_MD(REALV, REALH, true) \
  }
    if (d.real_vd) {
      if (d.real_h) HAMD_MD_P(true, true) else HAMD_MD_P(true, false)
    } else {
      if (d.real_h) HAMD_MD_P(false, true) else HAMD_MD_P(false, false)
    }
#undef HAMD_MD_P
#undef HAMD_MD
  });
  return grid;
}

}  // namespace

template <typename R, bool F64>
int launch_hilb_mfma(const FormDev& d, const StageArgs& A, hipStream_t st) {
  if (d.mfma == 2) {
    if constexpr (std::is_same<R, float>::value) {
      return d.tile == 32 ? launch_hilb_mfma_n<32, float, false, true>(d, A, st)
                          : launch_hilb_mfma_n<64, float, false, true>(d, A, st);
    } else {
      throw HeomError{HEOM_ERR_UNSUPPORTED, "bf16x3 products need the FP32 state"};
    }
  }
  if constexpr (std::is_same<R, double>::value)
    if (d.tile == 48) return launch_hilb_mfma_n<48, R, F64, false>(d, A, st);
  return d.tile == 32 ? launch_hilb_mfma_n<32, R, F64, false>(d, A, st)
                      : launch_hilb_mfma_n<64, R, F64, false>(d, A, st);
}

template <typename R, bool F64>
int launch_hilb_mfma_dense(const FormDev& d, const StageArgs& A, hipStream_t st) {
  return d.tile == 32   ? launch_hilb_mfma_dense_n<32, R, F64>(d, A, st)
         : d.tile == 48 ? launch_hilb_mfma_dense_n<48, R, F64>(d, A, st)
                        : launch_hilb_mfma_dense_n<64, R, F64>(d, A, st);
}

HAMD_FORM_INSTANCES(launch_hilb_mfma)
HAMD_FORM_INSTANCES(launch_hilb_mfma_dense)

}  // namespace hamd
