// Kernels and host code of the closure network (mlp.h).  Every reduction is
// done in a fixed order (no atomics), so training is reproducible run to run.
#include "mlp.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <string>

#include "kernels.h"

namespace hamd {

namespace {

typedef float mf_f4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// FP32 matrix products of the network on the f32 matrix cores (16x16x4, FP32
// accumulation): a 64 x 64 output tile per workgroup of four waves (2 x 2
// accumulators each), k in slices of 32 staged in two LDS buffers while the next
// four (weight gradients: two) are in flight in registers.  LDS strides 36 (k contiguous) and 80 (m or n
// contiguous): the 64 lanes of an operand read hit 64 distinct banks.
//
// The sizes are small (4096 rows x 256 units: 256 tiles, one per CU; 0.5 GFLOP,
// 4 us at the f32 matrix rate), so a launch is bound by its k chain.  A weight
// gradient has few tiles (16 at 256 x 256) and a long k (the rows): it is split
// over k (ksplit rows per workgroup), every part into its own slice of a
// partial buffer that grad_reduce_kernel adds up in order.
// Loss and gradient of 4096 rows of a 49-256-256-32 network: 4850 us with
// unsplit 64 x 64 vector-ALU products (820 us per weight gradient, 880 us per
// serial column sum); 203 us with one slice ahead (19 us per layer product, 10 us
// the sum of the gradient's parts) and the results copied back, 126 us here (16 us,
// 9 us, results written to pinned memory).
// ---------------------------------------------------------------------------
constexpr int kT = 64, kK = 32;
constexpr int kLdK = kK + 4, kLdM = kT + 16;

enum GemmEpi { EPI_PLAIN = 0, EPI_TANH = 1, EPI_TANH_BACK = 2, EPI_MSE = 3 };

// C[M x N] = op(A) op(B); op(A)(m, k) = TA ? A[k*lda + m] : A[m*lda + k], op(B) likewise
struct GemmArgs {
  int M, N, K;
  const float *A, *B;
  int lda, ldb, ldc;
  float* C;
  const float* bias;  // added per column (null: none)
  int epi;
  const float* H;     // EPI_TANH_BACK: C *= 1 - H^2 (the stored activation, ld = ldc)
  // EPI_MSE: T = normalised target rows; C = 2 (v - T) / (M N), the sum of
  // (v - T)^2 over the tile to loss[workgroup]
  const float *Y, *ym, *ys;
  const int* perm;
  double* loss;
  // split over k (weight gradients): part z of C starts at C + z * part_stride;
  // asum (null: none) receives the sums of op(A) over the part's k (bias gradient)
  int ksplit;
  long long part_stride;
  float* asum;
};

// four consecutive elements of a row of n (zero at and past n; p: the row)
__device__ __forceinline__ mf_f4 ld4(const float* p, int c, int n, bool vec) {
  if (vec && c + 4 <= n) return *reinterpret_cast<const mf_f4*>(p + c);
  mf_f4 v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (c + q < n) v[q] = p[c + q];
  return v;
}

// TR: the operand is stored k-major (rows of k), else m-major (rows of m).
// Thread tid takes two groups of four elements of the 64 x 32 slice at (m0, k0).
template <bool TR>
struct Slice {
  mf_f4 v[2];
  __device__ __forceinline__ void load(const float* P, int ld, int m0, int M, int k0, int k1,
                                       bool vec) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = threadIdx.x + 256 * i;
      const int r = TR ? k0 + x / 16 : m0 + x / 8;   // row in memory
      const int c = TR ? m0 + 4 * (x % 16) : k0 + 4 * (x % 8);
      const bool in = r < (TR ? k1 : M);
      v[i] = in ? ld4(P + static_cast<long long>(r) * ld, c, TR ? M : k1, vec)
                : mf_f4{0.f, 0.f, 0.f, 0.f};
    }
  }
  __device__ __forceinline__ void store(float* s) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = threadIdx.x + 256 * i;
      float* d = TR ? s + (x / 16) * kLdM + 4 * (x % 16) : s + (x / 8) * kLdK + 4 * (x % 8);
      *reinterpret_cast<mf_f4*>(d) = v[i];
    }
  }
};

template <bool TA, bool TB>
__device__ void gemm_tile(const GemmArgs& g, int bx, int by, int bz, int wg) {
  __shared__ __align__(16) float s_a[2][TA ? kK * kLdM : kT * kLdK];
  __shared__ __align__(16) float s_b[2][TB ? kT * kLdK : kK * kLdM];
  __shared__ double s_loss[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int m0 = by * kT, n0 = bx * kT;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int k0 = bz * g.ksplit, k1 = min(g.K, k0 + g.ksplit);
  const bool va = g.lda % 4 == 0 && (reinterpret_cast<uintptr_t>(g.A) & 15) == 0;
  const bool vb = g.ldb % 4 == 0 && (reinterpret_cast<uintptr_t>(g.B) & 15) == 0;
  mf_f4 acc[2][2] = {};
  float asum = 0.f;
  // k slices in flight in registers (even: two LDS buffers); a part of a weight
  // gradient has three workgroups per CU, which hide their loads already (four slices:
  // 17.5 -> 20 us)
  constexpr int kAhead = TA ? 2 : 4;
  Slice<TA> a[kAhead];
  Slice<!TB> b[kAhead];
  auto load = [&](int p, int k) {
    if (k >= k1) return;
    a[p].load(g.A, g.lda, m0, g.M, k, k1, va);
    b[p].load(g.B, g.ldb, n0, g.N, k, k1, vb);
  };
#pragma unroll
  for (int p = 0; p < kAhead; ++p) load(p, k0 + p * kK);
  for (int kb = k0; kb < k1; kb += kAhead * kK) {
#pragma unroll
    for (int p = 0; p < kAhead; ++p) {
      const int k = kb + p * kK;
      if (k >= k1) break;
      // two LDS buffers, one barrier: the slice before the last was read by
      // every wave before it reached the last barrier
      float *As = s_a[p & 1], *Bs = s_b[p & 1];
      a[p].store(As);
      b[p].store(Bs);
      __syncthreads();
      load(p, k + kAhead * kK);
#pragma unroll
      for (int s = 0; s < kK / 4; ++s) {
        const int kk = 4 * s + lk;
        float av[2], bv[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int m = wm + 16 * t + lr, n = wn + 16 * t + lr;
          av[t] = TA ? As[kk * kLdM + m] : As[m * kLdK + kk];
          bv[t] = TB ? Bs[n * kLdK + kk] : Bs[kk * kLdM + n];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
      }
      if (TA && g.asum && bx == 0 && threadIdx.x < kT)
        for (int kk = 0; kk < kK; ++kk) asum += As[kk * kLdM + threadIdx.x];
    }
  }
  if (TA && g.asum && bx == 0 && threadIdx.x < kT && m0 + static_cast<int>(threadIdx.x) < g.M)
    g.asum[bz * g.part_stride + m0 + threadIdx.x] = asum;
  float* C = g.C + bz * g.part_stride;
  double loss = 0.0;
  const float scale = 2.f / (static_cast<float>(g.M) * static_cast<float>(g.N));
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int m = m0 + wm + 16 * i + 4 * lk + q;
      if (m >= g.M) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn + 16 * j + lr;
        if (n >= g.N) continue;
        const long long at = static_cast<long long>(m) * g.ldc + n;
        float v = acc[i][j][q];
        if (g.bias) v += g.bias[n];
        if (g.epi == EPI_TANH) {
          v = tanhf(v);
        } else if (g.epi == EPI_TANH_BACK) {
          const float h = g.H[at];
          v *= 1.f - h * h;
        } else if (g.epi == EPI_MSE) {
          const long long r = g.perm ? g.perm[m] : m;
          const float d = v - (g.Y[r * g.N + n] - g.ym[n]) / g.ys[n];
          loss += static_cast<double>(d) * d;
          v = scale * d;
        }
        C[at] = v;
      }
    }
  if (g.epi == EPI_MSE) {
    for (int o = 32; o > 0; o >>= 1) loss += __shfl_down(loss, o, 64);
    if (lane == 0) s_loss[wave] = loss;
    __syncthreads();
    if (threadIdx.x == 0) g.loss[wg] = (s_loss[0] + s_loss[1]) + (s_loss[2] + s_loss[3]);
  }
}

template <bool TA, bool TB>
__global__ void __launch_bounds__(256) gemm_kernel(const GemmArgs g) {
  gemm_tile<TA, TB>(g, blockIdx.x, blockIdx.y, 0, blockIdx.y * gridDim.x + blockIdx.x);
}

// The three weight gradients (and bias gradients) of a backward pass in one
// launch: workgroups wg0[i] .. wg0[i+1] take the tiles and k parts of product i.
struct GradArgs {
  GemmArgs g[3];
  int wg0[4], nx[3], ny[3];
};

__global__ void __launch_bounds__(256) grad_kernel(const GradArgs a) {
  const int b = blockIdx.x;
  const int i = b >= a.wg0[2] ? 2 : b >= a.wg0[1] ? 1 : 0;
  const int r = b - a.wg0[i], nt = a.nx[i] * a.ny[i];
  const int z = r / nt, t = r - z * nt;
  gemm_tile<true, false>(a.g[i], t % a.nx[i], t / a.nx[i], z, b);
}

// grads[i] = sum over the parts, in order; workgroup 0 also adds up the loss
// partials (fixed order) and divides by their element count
// (out: host memory); host (may be null): the gradient in pinned host memory too
__global__ void __launch_bounds__(256) grad_reduce_kernel(const float* parts, int n_parts,
                                                          long long n, float* grads,
                                                          const double* loss, int n_loss,
                                                          double count, double* out,
                                                          float* host) {
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) {
    float s = 0.f;
    int p = 0;
    for (; p + 8 <= n_parts; p += 8) {  // eight parts in flight, added in order
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = parts[(p + q) * n + i];
#pragma unroll
      for (int q = 0; q < 8; ++q) s += v[q];
    }
    for (; p < n_parts; ++p) s += parts[p * n + i];
    grads[i] = s;
    if (host) host[i] = s;
  }
  if (blockIdx.x != 0) return;
  __shared__ double sd[256];
  double l = 0.0;
  for (int p = threadIdx.x; p < n_loss; p += 256) l += loss[p];
  sd[threadIdx.x] = l;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (static_cast<int>(threadIdx.x) < o) sd[threadIdx.x] += sd[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = sd[0] / count;
}

// Adam (Kingma & Ba, 2015) with bias-corrected moments
__global__ void adam_kernel(float* p, const float* g, float* m, float* v, long long n, float lr,
                            float b1, float b2, float eps, float c1, float c2) {
  for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<long long>(gridDim.x) * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// per-column mean and standard deviation over rows (two passes, fixed order);
// a constant column gets scale 1
__global__ void colstats_kernel(const float* X, long long rows, int cols, float* mean,
                                float* scale) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= cols) return;
  double s = 0.0;
  for (long long r = 0; r < rows; ++r) s += X[r * cols + j];
  const double mu = s / static_cast<double>(rows);
  double q = 0.0;
  for (long long r = 0; r < rows; ++r) {
    const double d = X[r * cols + j] - mu;
    q += d * d;
  }
  const double sd = sqrt(q / static_cast<double>(rows));
  mean[j] = static_cast<float>(mu);
  scale[j] = sd > 1e-30 * (fabs(mu) + 1e-30) && sd > 0.0 ? static_cast<float>(sd) : 1.f;
}

// normalised rows: out[r][j] = (X[perm[r] or r][j] - mean[j]) / scale[j]
__global__ void gather_norm_kernel(const float* X, const int* perm, int rows, int cols,
                                   const float* mean, const float* scale, float* out) {
  const long long n = static_cast<long long>(rows) * cols;
  for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<long long>(gridDim.x) * blockDim.x) {
    const int r = static_cast<int>(i / cols), j = static_cast<int>(i - static_cast<long long>(r) * cols);
    const long long src = perm ? perm[r] : r;
    out[i] = (X[src * cols + j] - mean[j]) / scale[j];
  }
}

// Y = Yn * scale + mean (column-wise)
__global__ void denorm_kernel(const float* Yn, int rows, int cols, const float* mean,
                              const float* scale, float* Y) {
  const long long n = static_cast<long long>(rows) * cols;
  for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<long long>(gridDim.x) * blockDim.x) {
    const int j = static_cast<int>(i % cols);
    Y[i] = Yn[i] * scale[j] + mean[j];
  }
}

// x: Re / Im blocks of the last-tier ADOs (ADO r at r * x_stride) and the
// constant columns; y: the dropped terms, y = -buf with
// buf = -D_full + D_trunc, in blocks of 2 N^2
__global__ void closure_pack_kernel(const z128* rho, const z128* buf, long long base, int n_ado,
                                    int N2, int x_stride, float* x, float* y, const float* cst,
                                    int cst_rows, int n_cst, int cst_off, int row_len) {
  const long long n = static_cast<long long>(n_ado) * N2;
  for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<long long>(gridDim.x) * blockDim.x) {
    const long long r = i / N2;
    const int e = static_cast<int>(i - r * N2);
    const z128 v = rho[base + i], b = buf[base + i];
    x[r * x_stride + e] = static_cast<float>(v.re);
    x[r * x_stride + N2 + e] = static_cast<float>(v.im);
    y[r * 2 * N2 + e] = static_cast<float>(-b.re);
    y[r * 2 * N2 + N2 + e] = static_cast<float>(-b.im);
  }
  const long long nc = static_cast<long long>(cst_rows) * n_cst;
  for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < nc;
       i += static_cast<long long>(gridDim.x) * blockDim.x) {
    const long long r = i / n_cst;
    x[r * row_len + cst_off + (i - r * n_cst)] = cst[i];
  }
}

int grid_for(long long n) {
  const long long g = (n + 255) / 256;
  return static_cast<int>(g < 4096 ? (g < 1 ? 1 : g) : 4096);
}

uint64_t splitmix(uint64_t& s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

double uniform01(uint64_t& s) { return (splitmix(s) >> 11) * (1.0 / 9007199254740992.0); }

}  // namespace

namespace {

GemmArgs gemm_args(int M, int N, int K, const float* A, int lda, const float* B, int ldb, float* C,
                   int ldc) {
  GemmArgs g{};
  g.M = M;
  g.N = N;
  g.K = K;
  g.A = A;
  g.B = B;
  g.lda = lda;
  g.ldb = ldb;
  g.C = C;
  g.ldc = ldc;
  g.ksplit = K;
  return g;
}

int gemm_tiles(int n) { return (n + kT - 1) / kT; }

template <bool TA, bool TB>
void launch_gemm(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.N <= 0) return;
  hipLaunchKernelGGL((gemm_kernel<TA, TB>), dim3(gemm_tiles(g.N), gemm_tiles(g.M)), dim3(256), 0,
                     st, g);
  HAMD_HIP(hipGetLastError());
}

}  // namespace

void launch_layer(int rows, int n_out, int n_in, const float* x, const float* W, const float* b,
                  float* y, bool act, hipStream_t st) {
  GemmArgs g = gemm_args(rows, n_out, n_in, x, n_in, W, n_in, y, n_out);
  g.bias = b;
  g.epi = act ? EPI_TANH : EPI_PLAIN;
  launch_gemm<false, true>(g, st);
}

// ---------------------------------------------------------------------------
// Mlp
// ---------------------------------------------------------------------------
Mlp::Mlp(int n_in_, int n_hidden, int n_out_, uint64_t seed, int device_)
    : n_in(n_in_), n_hid(n_hidden), n_out(n_out_), device(device_) {
  if (n_in < 1 || n_hid < 1 || n_out < 1)
    throw HeomError{HEOM_ERR_ARG, "mlp: layer sizes must be >= 1"};
  HAMD_HIP(hipSetDevice(device));
  HAMD_HIP(hipStreamCreate(&stream));
  n_par = static_cast<long long>(n_hid) * n_in + n_hid + static_cast<long long>(n_hid) * n_hid +
          n_hid + static_cast<long long>(n_out) * n_hid + n_out;
  // Glorot-uniform weights, zero biases
  std::vector<float> h(n_par, 0.f);
  uint64_t s = seed;
  auto fill = [&](long long off, int fan_out, int fan_in) {
    const double a = std::sqrt(6.0 / (fan_in + fan_out));
    for (long long i = 0; i < static_cast<long long>(fan_out) * fan_in; ++i)
      h[off + i] = static_cast<float>((2.0 * uniform01(s) - 1.0) * a);
  };
  long long o = 0;
  fill(o, n_hid, n_in);
  o += static_cast<long long>(n_hid) * n_in + n_hid;
  fill(o, n_hid, n_hid);
  o += static_cast<long long>(n_hid) * n_hid + n_hid;
  fill(o, n_out, n_hid);
  params.upload(h);
  std::vector<float> z(n_par, 0.f);
  grads.upload(z);
  adam_m.upload(z);
  adam_v.upload(z);
  std::vector<float> zi(n_in, 0.f), oi(n_in, 1.f), zo(n_out, 0.f), oo(n_out, 1.f);
  xm_.upload(zi);
  xs_.upload(oi);
  ym_.upload(zo);
  ys_.upload(oo);
}

Mlp::~Mlp() {
  if (stream) (void)hipStreamDestroy(stream);
  if (h_loss) (void)hipHostFree(h_loss);
  if (h_grad) (void)hipHostFree(h_grad);
}

float* Mlp::W1() const { return params.as<float>(); }
float* Mlp::b1() const { return W1() + static_cast<long long>(n_hid) * n_in; }
float* Mlp::W2() const { return b1() + n_hid; }
float* Mlp::b2() const { return W2() + static_cast<long long>(n_hid) * n_hid; }
float* Mlp::W3() const { return b2() + n_hid; }
float* Mlp::b3() const { return W3() + static_cast<long long>(n_out) * n_hid; }

void Mlp::get_params(float* host) const {
  HAMD_HIP(hipMemcpy(host, params.p, sizeof(float) * n_par, hipMemcpyDeviceToHost));
}

void Mlp::set_params(const float* host) {
  HAMD_HIP(hipMemcpy(params.p, host, sizeof(float) * n_par, hipMemcpyHostToDevice));
}

void Mlp::set_scaling(const float* xm, const float* xs, const float* ym, const float* ys) {
  for (int j = 0; j < n_in; ++j)
    if (!(xs[j] > 0.f)) throw HeomError{HEOM_ERR_ARG, "mlp: input scale must be > 0"};
  for (int j = 0; j < n_out; ++j)
    if (!(ys[j] > 0.f)) throw HeomError{HEOM_ERR_ARG, "mlp: output scale must be > 0"};
  HAMD_HIP(hipMemcpy(xm_.p, xm, sizeof(float) * n_in, hipMemcpyHostToDevice));
  HAMD_HIP(hipMemcpy(xs_.p, xs, sizeof(float) * n_in, hipMemcpyHostToDevice));
  HAMD_HIP(hipMemcpy(ym_.p, ym, sizeof(float) * n_out, hipMemcpyHostToDevice));
  HAMD_HIP(hipMemcpy(ys_.p, ys, sizeof(float) * n_out, hipMemcpyHostToDevice));
}

void Mlp::get_scaling(float* xm, float* xs, float* ym, float* ys) const {
  if (xm) HAMD_HIP(hipMemcpy(xm, xm_.p, sizeof(float) * n_in, hipMemcpyDeviceToHost));
  if (xs) HAMD_HIP(hipMemcpy(xs, xs_.p, sizeof(float) * n_in, hipMemcpyDeviceToHost));
  if (ym) HAMD_HIP(hipMemcpy(ym, ym_.p, sizeof(float) * n_out, hipMemcpyDeviceToHost));
  if (ys) HAMD_HIP(hipMemcpy(ys, ys_.p, sizeof(float) * n_out, hipMemcpyDeviceToHost));
}

void Mlp::fit_scaling(const float* X, const float* Y, long long n_rows) {
  if (n_rows < 1) throw HeomError{HEOM_ERR_ARG, "mlp: no rows"};
  HAMD_HIP(hipSetDevice(device));
  hipLaunchKernelGGL(colstats_kernel, dim3((n_in + 255) / 256), dim3(256), 0, stream, X, n_rows,
                     n_in, xm_.as<float>(), xs_.as<float>());
  hipLaunchKernelGGL(colstats_kernel, dim3((n_out + 255) / 256), dim3(256), 0, stream, Y, n_rows,
                     n_out, ym_.as<float>(), ys_.as<float>());
  HAMD_HIP(hipGetLastError());
  HAMD_HIP(hipStreamSynchronize(stream));
}

// k parts of the weight gradients: parts of 128 rows (four k slices) give the
// 256 x 256 gradient 16 tiles x 32 parts at 4096 rows, two workgroups per CU; at
// most 64 parts, and at most 64 MB of partial gradients (a network with more
// parameters than that allows fills the chip with fewer parts).
int Mlp::max_grad_parts() const {
  const long long fit = (64LL << 20) / static_cast<long long>(sizeof(float)) / n_par;
  return static_cast<int>(std::max(1LL, std::min(64LL, fit)));
}

int Mlp::grad_split(int rows) const {
  constexpr int kMin = 4;  // k slices per part
  const int slices = (rows + kK - 1) / kK, cap = max_grad_parts();
  return std::max(kMin, (slices + cap - 1) / cap) * kK;
}

void Mlp::ensure_rows(int rows) {
  if (rows <= cap_rows) return;
  xb.alloc(sizeof(float) * rows * static_cast<size_t>(n_in));
  h1.alloc(sizeof(float) * rows * static_cast<size_t>(n_hid));
  h2.alloc(sizeof(float) * rows * static_cast<size_t>(n_hid));
  dh1.alloc(sizeof(float) * rows * static_cast<size_t>(n_hid));
  dh2.alloc(sizeof(float) * rows * static_cast<size_t>(n_hid));
  yb.alloc(sizeof(float) * rows * static_cast<size_t>(n_out));
  dyb.alloc(sizeof(float) * rows * static_cast<size_t>(n_out));
  partials.alloc(sizeof(double) * gemm_tiles(n_out) * gemm_tiles(rows));
  cap_rows = rows;
}

void Mlp::forward_hidden(int rows) {
  launch_layer(rows, n_hid, n_in, xb.as<float>(), W1(), b1(), h1.as<float>(), true, stream);
  launch_layer(rows, n_hid, n_hid, h1.as<float>(), W2(), b2(), h2.as<float>(), true, stream);
}

void Mlp::forward(const float* X, float* Y, int n_rows) {
  HAMD_HIP(hipSetDevice(device));
  const int chunk = 8192;
  for (int r0 = 0; r0 < n_rows; r0 += chunk) {
    const int rows = std::min(chunk, n_rows - r0);
    ensure_rows(rows);
    hipLaunchKernelGGL(gather_norm_kernel, dim3(grid_for(static_cast<long long>(rows) * n_in)),
                       dim3(256), 0, stream, X + static_cast<long long>(r0) * n_in,
                       static_cast<const int*>(nullptr), rows, n_in, xm_.as<float>(),
                       xs_.as<float>(), xb.as<float>());
    forward_hidden(rows);
    launch_layer(rows, n_out, n_hid, h2.as<float>(), W3(), b3(), yb.as<float>(), false, stream);
    hipLaunchKernelGGL(denorm_kernel, dim3(grid_for(static_cast<long long>(rows) * n_out)),
                       dim3(256), 0, stream, yb.as<float>(), rows, n_out, ym_.as<float>(),
                       ys_.as<float>(), Y + static_cast<long long>(r0) * n_out);
    HAMD_HIP(hipGetLastError());
  }
  HAMD_HIP(hipStreamSynchronize(stream));
}

// Forward, loss and gradient in eight launches (the gather, three layers with
// the loss in the last one's epilogue, two backward products with the
// derivative of tanh in theirs, the weight and bias gradients, their sum).
// Loss and, on request, gradient come back through pinned host memory that the last
// kernel writes: one synchronisation and no copy commands.
double Mlp::loss_grad(const float* X, const float* Y, int rows, const int* perm_dev,
                      float* grad_host) {
  HAMD_HIP(hipSetDevice(device));
  ensure_rows(rows);
  if (h_loss == nullptr)
    HAMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&h_loss), 64, hipHostMallocCoherent));
  if (grad_host && h_grad == nullptr)
    HAMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&h_grad), sizeof(float) * n_par,
                           hipHostMallocCoherent));
  const long long ni = static_cast<long long>(rows) * n_in, no = static_cast<long long>(rows) * n_out;
  hipLaunchKernelGGL(gather_norm_kernel, dim3(grid_for(ni)), dim3(256), 0, stream, X, perm_dev,
                     rows, n_in, xm_.as<float>(), xs_.as<float>(), xb.as<float>());
  forward_hidden(rows);
  // layer 3: dY = 2 (yhat - t) / n and the loss partials, one per tile
  GemmArgs f = gemm_args(rows, n_out, n_hid, h2.as<float>(), n_hid, W3(), n_hid, dyb.as<float>(),
                         n_out);
  f.bias = b3();
  f.epi = EPI_MSE;
  f.Y = Y;
  f.ym = ym_.as<float>();
  f.ys = ys_.as<float>();
  f.perm = perm_dev;
  f.loss = partials.as<double>();
  const int n_loss = gemm_tiles(n_out) * gemm_tiles(rows);
  launch_gemm<false, true>(f, stream);
  // dH2 = dY W3 (1 - h2^2), dH1 = dH2 W2 (1 - h1^2)
  GemmArgs b = gemm_args(rows, n_hid, n_out, dyb.as<float>(), n_out, W3(), n_hid, dh2.as<float>(),
                         n_hid);
  b.epi = EPI_TANH_BACK;
  b.H = h2.as<float>();
  launch_gemm<false, false>(b, stream);
  b = gemm_args(rows, n_hid, n_hid, dh2.as<float>(), n_hid, W2(), n_hid, dh1.as<float>(), n_hid);
  b.epi = EPI_TANH_BACK;
  b.H = h1.as<float>();
  launch_gemm<false, false>(b, stream);
  // gradients, laid out as the parameters, one slice per k part
  const int split = grad_split(rows), n_parts = (rows + split - 1) / split;
  const size_t gbytes = sizeof(float) * n_par * static_cast<size_t>(n_parts);
  if (gparts.bytes < gbytes) gparts.alloc(gbytes);
  float* gp = gparts.as<float>();
  float* pW1 = gp;
  float* pb1 = pW1 + static_cast<long long>(n_hid) * n_in;
  float* pW2 = pb1 + n_hid;
  float* pb2 = pW2 + static_cast<long long>(n_hid) * n_hid;
  float* pW3 = pb2 + n_hid;
  float* pb3 = pW3 + static_cast<long long>(n_out) * n_hid;
  GradArgs ga{};
  ga.g[0] = gemm_args(n_hid, n_hid, rows, dh2.as<float>(), n_hid, h1.as<float>(), n_hid, pW2, n_hid);
  ga.g[0].asum = pb2;
  ga.g[1] = gemm_args(n_hid, n_in, rows, dh1.as<float>(), n_hid, xb.as<float>(), n_in, pW1, n_in);
  ga.g[1].asum = pb1;
  ga.g[2] = gemm_args(n_out, n_hid, rows, dyb.as<float>(), n_out, h2.as<float>(), n_hid, pW3, n_hid);
  ga.g[2].asum = pb3;
  for (int i = 0; i < 3; ++i) {
    ga.g[i].ksplit = split;
    ga.g[i].part_stride = n_par;
    ga.nx[i] = gemm_tiles(ga.g[i].N);
    ga.ny[i] = gemm_tiles(ga.g[i].M);
    ga.wg0[i + 1] = ga.wg0[i] + ga.nx[i] * ga.ny[i] * n_parts;
  }
  hipLaunchKernelGGL(grad_kernel, dim3(ga.wg0[3]), dim3(256), 0, stream, ga);
  hipLaunchKernelGGL(grad_reduce_kernel, dim3(static_cast<int>((n_par + 255) / 256)), dim3(256), 0,
                     stream, gp, n_parts, n_par, grads.as<float>(), partials.as<double>(), n_loss,
                     static_cast<double>(no), h_loss, grad_host ? h_grad : nullptr);
  HAMD_HIP(hipGetLastError());
  HAMD_HIP(hipStreamSynchronize(stream));
  if (grad_host) std::memcpy(grad_host, h_grad, sizeof(float) * n_par);
  return *h_loss;
}

void Mlp::adam_step(double lr, double beta1, double beta2, double eps) {
  HAMD_HIP(hipSetDevice(device));
  t_adam += 1;
  const float c1 = static_cast<float>(1.0 - std::pow(beta1, static_cast<double>(t_adam)));
  const float c2 = static_cast<float>(1.0 - std::pow(beta2, static_cast<double>(t_adam)));
  hipLaunchKernelGGL(adam_kernel, dim3(grid_for(n_par)), dim3(256), 0, stream, params.as<float>(),
                     grads.as<float>(), adam_m.as<float>(), adam_v.as<float>(), n_par,
                     static_cast<float>(lr), static_cast<float>(beta1), static_cast<float>(beta2),
                     static_cast<float>(eps), c1, c2);
  HAMD_HIP(hipGetLastError());
}

void Mlp::train(const float* X, const float* Y, long long n_rows, int batch, int epochs,
                double lr, uint64_t seed, double* epoch_loss) {
  if (n_rows < 1 || batch < 1 || epochs < 0)
    throw HeomError{HEOM_ERR_ARG, "mlp train: bad sizes"};
  if (n_rows > (1LL << 31) - 1) throw HeomError{HEOM_ERR_UNSUPPORTED, "mlp train: too many rows"};
  HAMD_HIP(hipSetDevice(device));
  std::vector<int> order(static_cast<size_t>(n_rows));
  perm.alloc(sizeof(int) * order.size());
  uint64_t s = seed;
  for (int ep = 0; ep < epochs; ++ep) {
    std::iota(order.begin(), order.end(), 0);
    for (long long i = n_rows - 1; i > 0; --i) {  // Fisher-Yates
      const long long j = static_cast<long long>(splitmix(s) % static_cast<uint64_t>(i + 1));
      std::swap(order[i], order[j]);
    }
    HAMD_HIP(hipMemcpyAsync(perm.p, order.data(), sizeof(int) * order.size(),
                            hipMemcpyHostToDevice, stream));
    double tot = 0.0;
    for (long long r0 = 0; r0 < n_rows; r0 += batch) {
      const int rows = static_cast<int>(std::min<long long>(batch, n_rows - r0));
      tot += loss_grad(X, Y, rows, perm.as<int>() + r0) * rows;
      adam_step(lr, 0.9, 0.999, 1e-8);
    }
    if (epoch_loss) epoch_loss[ep] = tot / static_cast<double>(n_rows);
  }
  HAMD_HIP(hipStreamSynchronize(stream));
}

// ---------------------------------------------------------------------------
// Closure
// ---------------------------------------------------------------------------
void last_tier(const Qme& q, int& first, int& count) {
  const int K = q.hs.n_dim;
  first = q.hs.n_hrchy;
  for (int a = 0; a < q.hs.n_hrchy; ++a) {
    int tier = 0;
    for (int k = 0; k < K; ++k) tier += q.hs.n[static_cast<size_t>(a) * K + k];
    if (tier == q.max_depth) {
      first = a;
      break;
    }
  }
  count = q.hs.n_hrchy - first;  // breadth-first order: the last tier is a suffix
}

ClosureDims closure_dims(const Qme& q, int layout, int n_features) {
  if (layout != HEOM_CLOSURE_PER_ADO && layout != HEOM_CLOSURE_GLOBAL)
    throw HeomError{HEOM_ERR_ARG, "closure: unknown layout"};
  if (n_features < 0) throw HeomError{HEOM_ERR_ARG, "closure: n_features < 0"};
  ClosureDims c{};
  last_tier(q, c.lo, c.n_ado);
  const int K = q.hs.n_dim, N2 = q.N2;
  if (layout == HEOM_CLOSURE_PER_ADO) {
    c.rows = c.n_ado;
    c.n_in = 2 * N2 + K + n_features;
    c.n_out = 2 * N2;
    c.ado_stride = c.n_in;
    c.cst_rows = c.n_ado;
    c.n_cst = K + n_features;
    c.cst_off = 2 * N2;
  } else {
    c.rows = 1;
    c.n_in = 2 * N2 * c.n_ado + n_features;
    c.n_out = 2 * N2 * c.n_ado;
    c.ado_stride = 2 * N2;
    c.cst_rows = 1;
    c.n_cst = n_features;
    c.cst_off = 2 * N2 * c.n_ado;
  }
  return c;
}

namespace {
// constant input columns of a closure row buffer: index vectors and features
std::vector<float> closure_constants(const Qme& q, const ClosureDims& c, int layout,
                                     const float* features, int n_features) {
  const int K = q.hs.n_dim;
  std::vector<float> cst(static_cast<size_t>(c.cst_rows) * c.n_cst);
  for (int r = 0; r < c.cst_rows; ++r) {
    float* row = cst.data() + static_cast<size_t>(r) * c.n_cst;
    int o = 0;
    if (layout == HEOM_CLOSURE_PER_ADO)
      for (int k = 0; k < K; ++k)
        row[o++] = static_cast<float>(q.hs.n[static_cast<size_t>(c.lo + r) * K + k]);
    for (int f = 0; f < n_features; ++f) row[o++] = features[f];
  }
  return cst;
}
}  // namespace

void closure_rows(Qme& deep, Qme& shallow, const void* rho_deep, const float* features,
                  int n_features, int layout, float* x, float* y) {
  if (deep.kind != HEOM_HILB || shallow.kind != HEOM_HILB)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "closure rows: heom_hilb only"};
  if (deep.lo() || shallow.lo())
    throw HeomError{HEOM_ERR_ARG, "closure rows: both QMEs must be complex128"};
  if (deep.N != shallow.N || deep.hs.n_dim != shallow.hs.n_dim ||
      shallow.max_depth >= deep.max_depth || shallow.max_depth < 1)
    throw HeomError{HEOM_ERR_ARG, "closure rows: shallow must be the same model at a smaller "
                                  "depth >= 1"};
  // the shallow hierarchy must be a prefix of the deep one (breadth-first order)
  for (size_t i = 0; i < shallow.hs.n.size(); ++i)
    if (shallow.hs.n[i] != deep.hs.n[i])
      throw HeomError{HEOM_ERR_ARG, "closure rows: hierarchies differ"};
  if (n_features > 0 && !features) throw HeomError{HEOM_ERR_ARG, "closure rows: bad features"};
  const ClosureDims c = closure_dims(shallow, layout, n_features);
  const int N2 = shallow.N2;
  HAMD_HIP(hipSetDevice(deep.opt.device));
  hipStream_t st = deep.stream;
  HAMD_HIP(hipStreamSynchronize(shallow.stream));
  const size_t bytes = sizeof(z128) * static_cast<size_t>(deep.main_size());
  if (deep.scratch.bytes != bytes) deep.scratch.alloc(bytes);
  // buf = -D_full(rho); buf[shallow] += D_trunc(rho[shallow])
  const StageArgs a1 = deep.diff_args(deep.scratch.p, rho_deep, z128{1.0, 0.0}, z128{0.0, 0.0});
  launch_operator(deep.dev, 8, a1, st);
  const StageArgs a2 =
      shallow.diff_args(deep.scratch.p, rho_deep, z128{-1.0, 0.0}, z128{1.0, 0.0});
  launch_operator(shallow.dev, 8, a2, st);
  DevBuf dc;
  dc.upload(closure_constants(shallow, c, layout, features, n_features));
  const long long n = std::max(static_cast<long long>(c.n_ado) * N2,
                               static_cast<long long>(c.cst_rows) * c.n_cst);
  hipLaunchKernelGGL(closure_pack_kernel, dim3(grid_for(n)), dim3(256), 0, st,
                     static_cast<const z128*>(rho_deep), deep.scratch.as<z128>(),
                     static_cast<long long>(c.lo) * N2, c.n_ado, N2, c.ado_stride, x, y,
                     dc.as<float>(), c.cst_rows, c.n_cst, c.cst_off, c.n_in);
  HAMD_HIP(hipGetLastError());
  HAMD_HIP(hipStreamSynchronize(st));
}

namespace {
// a row-major n x k weight matrix, padded with zeros to np x kp, in the operand
// order of closure_mlp_kernel (see ClosureNet)
std::vector<float> operand_order(const std::vector<float>& w, int n, int k, int np, int kp) {
  std::vector<float> o(static_cast<size_t>(np) * kp, 0.f);
  for (int a = 0; a < n; ++a)
    for (int b = 0; b < k; ++b)
      o[((static_cast<size_t>(a / 16) * (kp / 16) + b / 16) * 64 + (b % 16) / 4 * 16 + a % 16) * 4 +
        b % 4] = w[static_cast<size_t>(a) * k + b];
  return o;
}
}  // namespace

void Closure::bind(Qme& q, const Mlp& m, const float* features, int n_features, int layout) {
  if (q.kind != HEOM_HILB)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "closure: heom_hilb only"};
  if (q.max_depth < 1) throw HeomError{HEOM_ERR_ARG, "closure: max_depth must be >= 1"};
  if (n_features > 0 && !features) throw HeomError{HEOM_ERR_ARG, "closure: bad features"};
  dm = closure_dims(q, layout, n_features);
  if (dm.n_ado < 1) throw HeomError{HEOM_ERR_ARG, "closure: no ADO at the last tier"};
  const int n_in = dm.n_in, n_out = dm.n_out;
  n_hid = m.n_hid;
  if (m.n_in != n_in || m.n_out != n_out)
    throw HeomError{HEOM_ERR_ARG, "closure: this layout needs a network with n_in = " +
                                      std::to_string(n_in) + " and n_out = " +
                                      std::to_string(n_out)};
  // fold the normalisation into the first and last layers
  std::vector<float> p(m.n_params()), xm(n_in), xs(n_in), ym(n_out), ys(n_out);
  m.get_params(p.data());
  m.get_scaling(xm.data(), xs.data(), ym.data(), ys.data());
  const long long oW1 = 0, ob1 = oW1 + static_cast<long long>(n_hid) * n_in, oW2 = ob1 + n_hid,
                  ob2 = oW2 + static_cast<long long>(n_hid) * n_hid, oW3 = ob2 + n_hid,
                  ob3 = oW3 + static_cast<long long>(n_out) * n_hid;
  std::vector<float> w1(static_cast<size_t>(n_hid) * n_in), bb1(n_hid),
      w3(static_cast<size_t>(n_out) * n_hid), bb3(n_out);
  for (int j = 0; j < n_hid; ++j) {
    double b = p[ob1 + j];
    for (int i = 0; i < n_in; ++i) {
      const double w = p[oW1 + static_cast<long long>(j) * n_in + i];
      w1[static_cast<size_t>(j) * n_in + i] = static_cast<float>(w / xs[i]);
      b -= w * xm[i] / xs[i];
    }
    bb1[j] = static_cast<float>(b);
  }
  for (int o = 0; o < n_out; ++o) {
    for (int j = 0; j < n_hid; ++j)
      w3[static_cast<size_t>(o) * n_hid + j] =
          p[oW3 + static_cast<long long>(o) * n_hid + j] * ys[o];
    bb3[o] = p[ob3 + o] * ys[o] + ym[o];
  }
  const std::vector<float> w2(p.begin() + oW2, p.begin() + ob2),
      bb2(p.begin() + ob2, p.begin() + oW3);
  HAMD_HIP(hipSetDevice(q.opt.device));
  // per-ADO rows of a network that fits: one fused launch per operator pass
  fused = layout == HEOM_CLOSURE_PER_ADO && closure_mlp_fits(n_in, n_hid, n_out);
  net = ClosureNet{};
  if (fused) {
    auto pad16 = [](int n) { return (n + 15) / 16 * 16; };
    net.n_in = n_in;
    net.n_out = n_out;
    net.in_pad = pad16(n_in);
    net.hid = pad16(n_hid);
    net.out_pad = pad16(n_out);
    net.parts = closure_mlp_parts(dm.rows, net.hid);
    auto bias = [](std::vector<float> b, int n) {
      b.resize(n, 0.f);
      return b;
    };
    W1.upload(operand_order(w1, n_hid, n_in, net.hid, net.in_pad));
    W2.upload(operand_order(w2, n_hid, n_hid, net.hid, net.hid));
    W3.upload(operand_order(w3, n_out, n_hid, net.out_pad, net.hid));
    b1.upload(bias(bb1, net.hid));
    b2.upload(bias(bb2, net.hid));
    b3.upload(bias(bb3, net.out_pad));
  } else {
    W1.upload(w1);
    b1.upload(bb1);
    W2.upload(w2);
    b2.upload(bb2);
    W3.upload(w3);
    b3.upload(bb3);
  }
  // the constant input columns are written once
  std::vector<float> xh(static_cast<size_t>(dm.rows) * n_in, 0.f);
  const std::vector<float> cst = closure_constants(q, dm, layout, features, n_features);
  for (int r = 0; r < dm.cst_rows; ++r)
    for (int c = 0; c < dm.n_cst; ++c)
      xh[static_cast<size_t>(r) * n_in + dm.cst_off + c] = cst[static_cast<size_t>(r) * dm.n_cst + c];
  x.upload(xh);
  if (!fused) {
    h1.alloc(sizeof(float) * dm.rows * static_cast<size_t>(n_hid));
    h2.alloc(sizeof(float) * dm.rows * static_cast<size_t>(n_hid));
  }
  const int parts = fused ? net.parts : 1;
  y.upload(std::vector<float>(static_cast<size_t>(parts) * dm.rows * n_out, 0.f));
  q.dev.clos = y.as<float>();
  q.dev.clos_lo = dm.lo;
  q.dev.clos_n = dm.n_ado;
  q.dev.clos_parts = parts;
  net.x = x.as<float>();
  net.W1 = W1.as<float>();
  net.b1 = b1.as<float>();
  net.W2 = W2.as<float>();
  net.b2 = b2.as<float>();
  net.W3 = W3.as<float>();
  net.b3 = b3.as<float>();
  net.y = y.as<float>();
}

void Closure::forward(const Qme& q, const StageArgs& A, hipStream_t st) {
  const int n_in = dm.n_in, n_out = dm.n_out, rows = dm.rows;
  if (fused) {
    launch_closure_mlp(q.dev, A, net, st);
    return;
  }
  launch_closure_gather(q.dev, A, x.as<float>(), dm.ado_stride, st);
  launch_layer(rows, n_hid, n_in, x.as<float>(), W1.as<float>(), b1.as<float>(), h1.as<float>(),
               true, st);
  launch_layer(rows, n_hid, n_hid, h1.as<float>(), W2.as<float>(), b2.as<float>(), h2.as<float>(),
               true, st);
  launch_layer(rows, n_out, n_hid, h2.as<float>(), W3.as<float>(), b3.as<float>(), y.as<float>(),
               false, st);
}

}  // namespace hamd
