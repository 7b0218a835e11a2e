// Inference of the learned truncation closure, one launch per operator pass.
#include "forms.h"
#include "stage.h"

namespace hamd {

namespace {

// closure network input (Re, Im of the last-tier ADOs of the stage input)
__global__ void closure_gather_kernel(const FormDev d, const StageArgs A, float* x,
                                      int ado_stride) {
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const void* in = pick(A.in, pg.cur);
  const long long n = static_cast<long long>(d.clos_n) * d.N2;
  const long long base = static_cast<long long>(d.clos_lo) * d.N2;
  for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<long long>(gridDim.x) * blockDim.x) {
    const z128 v = ldz(in, A.in_lo != 0, base + i);
    const long long r = i / d.N2;
    const int e = static_cast<int>(i - r * d.N2);
    x[r * ado_stride + e] = static_cast<float>(v.re);
    x[r * ado_stride + d.N2 + e] = static_cast<float>(v.im);
  }
}

// ---------------------------------------------------------------------------
// Learned closure, one launch per operator pass (per-ADO layout): each
// workgroup takes 16 last-tier ADOs of the stage input, gathers their network
// rows (Re, Im of rho_n, then the constant columns written at binding), and
// runs the three layers on the matrix cores (f32 16x16x4, FP32 accumulation):
// h1 = tanh(x W1^T + b1), h2 = tanh(h1 W2^T + b2), y = h2 W3^T + b3 (the
// normalisation folded into W1, b1, W3, b3).  Rows stay in LDS between layers.
//
// A small system has few rows (120 at four sites and depth 3: eight workgroups
// on 256 CUs), so the launch is a chain of latencies and the matrix pipe of one
// CU (16 x 256 x 256 products: 3.4 us).  The weights are therefore stored in
// operand order (one 16-byte load per lane covers four k steps, 1 KB per
// wavefront) and loaded before the rows are there; sixteen wavefronts share a
// layer's tiles, splitting k where it has fewer than sixteen; and `parts`
// workgroups share a row block: each runs layer 1, its share of the units of
// layer 2 and layer 3 on those, and the operator kernels add the partial
// outputs (parts 4 up to 64 row blocks, 2 up to 128: past that the rows fill
// the chip).  120 rows of a 49-256-256-32 network: 45 -> 9.7 us per pass.
// ---------------------------------------------------------------------------
constexpr int kClosRows = 16;    // network rows per workgroup
constexpr int kClosInMax = 128;  // widest input and output of the fused kernel
constexpr int kClosHidMax = 256;
constexpr int kClosWaves = 16;
constexpr int kClosPre = 4;      // k groups of 16 whose weights are loaded ahead

// One wavefront's share of a layer of T tiles of 16 units and KG k groups of 16:
// tile `tile`, groups [g0, g1) (none: tile < 0), S wavefronts per tile.
struct ClosJob {
  int tile, g0, g1, S;
  __device__ __forceinline__ ClosJob(int T, int KG, int wave) {
    S = 1;
    while (2 * S * T <= kClosWaves && 2 * S <= KG) S *= 2;
    tile = wave / S;
    const int per = (KG + S - 1) / S;
    g0 = (wave - tile * S) * per;
    g1 = min(KG, g0 + per);
    if (tile >= T || g0 >= g1) g1 = g0;
    if (tile >= T) tile = -1;
  }
};

// weights of k groups g0 .. g0 + kClosPre - 1 of the wavefront's tile; W: the
// layer in operand order, KGW groups per tile, from tile0 / group0 on
__device__ __forceinline__ void clos_prefetch(const ClosJob& j, const mf_f4* W, int KGW, int tile0,
                                              int group0, int lane, mf_f4 (&w)[kClosPre]) {
#pragma unroll
  for (int p = 0; p < kClosPre; ++p)
    if (j.g0 + p < j.g1)
      w[p] = W[(static_cast<long long>(tile0 + j.tile) * KGW + group0 + j.g0 + p) * 64 + lane];
}

// the layer: a (16 rows, leading dimension lda) times the weights into the
// partial sums red, then out(row, col, value) for every row and column
template <class Out>
__device__ __forceinline__ void clos_layer(const ClosJob& j, const float* a, int lda,
                                           const mf_f4* W, int KGW, int tile0, int group0, int T,
                                           const mf_f4 (&w)[kClosPre], mf_f4* red, Out out) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  if (j.tile >= 0) {
    // two accumulators: consecutive products do not wait for each other
    mf_f4 acc[2] = {mf_f4{0.f, 0.f, 0.f, 0.f}, mf_f4{0.f, 0.f, 0.f, 0.f}};
    for (int g = j.g0; g < j.g1; g += kClosPre) {
#pragma unroll
      for (int p = 0; p < kClosPre; ++p) {
        if (g + p < j.g1) {
          const mf_f4 b =
              g == j.g0 ? w[p]
                        : W[(static_cast<long long>(tile0 + j.tile) * KGW + group0 + g + p) * 64 +
                            lane];
          const mf_f4 v = *reinterpret_cast<const mf_f4*>(a + lr * lda + 16 * (g + p) + 4 * lk);
#pragma unroll
          for (int t = 0; t < 4; ++t)
            acc[t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t], b[t], acc[t & 1], 0, 0, 0);
        }
      }
    }
    red[wave * 64 + lane] = acc[0] + acc[1];
  }
  __syncthreads();
  const float* r = reinterpret_cast<const float*>(red);
  for (int x = threadIdx.x; x < 256 * T; x += 64 * kClosWaves) {
    const int tile = x >> 8, e = x & 255;
    float v = 0.f;
    for (int k = 0; k < j.S; ++k) v += r[(tile * j.S + k) * 256 + e];
    const int l = e >> 2;
    out(4 * (l >> 4) + (e & 3), 16 * tile + (l & 15), v);
  }
  __syncthreads();
}

__global__ void __launch_bounds__(64 * kClosWaves) closure_mlp_kernel(const FormDev d,
                                                                      const StageArgs A,
                                                                      const ClosureNet n) {
  constexpr int LDX = kClosInMax + 4, LDH = kClosHidMax + 4;
  __shared__ __align__(16) float s_x[kClosRows * LDX];
  __shared__ __align__(16) float s_h1[kClosRows * LDH];
  __shared__ __align__(16) float s_h2[kClosRows * LDH];
  __shared__ __align__(16) mf_f4 s_red[kClosWaves * 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int part = blockIdx.x % n.parts, r0 = (blockIdx.x / n.parts) * kClosRows;
  const int T1 = n.hid / 16, T2 = T1 / n.parts, T3 = n.out_pad / 16, KG1 = n.in_pad / 16;
  const mf_f4 *W1 = reinterpret_cast<const mf_f4*>(n.W1), *W2 = reinterpret_cast<const mf_f4*>(n.W2),
              *W3 = reinterpret_cast<const mf_f4*>(n.W3);
  const ClosJob j1(T1, KG1, wave), j2(T2, T1, wave), j3(T3, T2, wave);
  mf_f4 w1[kClosPre], w2[kClosPre], w3[kClosPre];
  clos_prefetch(j1, W1, KG1, 0, 0, lane, w1);
  clos_prefetch(j2, W2, T1, part * T2, 0, lane, w2);
  clos_prefetch(j3, W3, T1, 0, part * T2, lane, w3);
  const Prologue pg = prologue(A);
  if (pg.skip) return;
  const void* in = pick(A.in, pg.cur);
  const int rows = d.clos_n, N2 = d.N2;
  // gather: rho of ADO lo + r, then the constant columns (zero past n_in and rows)
  for (int x = threadIdx.x; x < kClosRows * n.in_pad; x += 64 * kClosWaves) {
    const int r = x / n.in_pad, c = x - r * n.in_pad;
    float v = 0.f;
    if (r0 + r < rows && c < n.n_in) {
      if (c < 2 * N2) {
        const z128 z = ldz(in, A.in_lo != 0,
                           At(static_cast<long long>(d.clos_lo + r0 + r) * N2,
                              c < N2 ? c : c - N2));
        v = static_cast<float>(c < N2 ? z.re : z.im);
      } else {
        v = n.x[static_cast<long long>(r0 + r) * n.n_in + c];
      }
    }
    s_x[r * LDX + c] = v;
  }
  __syncthreads();
  clos_layer(j1, s_x, LDX, W1, KG1, 0, 0, T1, w1, s_red, [&](int r, int c, float v) {
    s_h1[r * LDH + c] = tanhf(v + n.b1[c]);
  });
  clos_layer(j2, s_h1, LDH, W2, T1, part * T2, 0, T2, w2, s_red, [&](int r, int c, float v) {
    s_h2[r * LDH + c] = tanhf(v + n.b2[part * T2 * 16 + c]);
  });
  clos_layer(j3, s_h2, LDH, W3, T1, 0, part * T2, T3, w3, s_red, [&](int r, int c, float v) {
    if (c < n.n_out && r0 + r < rows)
      n.y[(static_cast<long long>(part) * rows + r0 + r) * n.n_out + c] =
          part == 0 ? v + n.b3[c] : v;
  });
}

}  // namespace

void launch_closure_gather(const FormDev& d, const StageArgs& A, float* x, int ado_stride,
                           hipStream_t stream) {
  const long long n = static_cast<long long>(d.clos_n) * d.N2;
  hipLaunchKernelGGL(closure_gather_kernel, dim3(cap_grid((n + 255) / 256)), dim3(256), 0, stream,
                     d, A, x, ado_stride);
  HAMD_HIP(hipGetLastError());
}

bool closure_mlp_fits(int n_in, int n_hid, int n_out) {
  return n_in <= kClosInMax && n_hid <= kClosHidMax && n_out <= kClosInMax;
}

int closure_mlp_parts(int rows, int hid_pad) {
  const int blocks = (rows + kClosRows - 1) / kClosRows, tiles = hid_pad / 16;
  if (blocks <= 64 && tiles % 4 == 0) return 4;
  return blocks <= 128 && tiles % 2 == 0 ? 2 : 1;
}

void launch_closure_mlp(const FormDev& d, const StageArgs& A, const ClosureNet& n,
                        hipStream_t stream) {
  if (!closure_mlp_fits(n.n_in, n.hid, n.n_out) || n.in_pad % 16 || n.hid % 16 || n.out_pad % 16 ||
      n.parts < 1 || (n.hid / 16) % n.parts)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "closure: network too wide for the fused kernel"};
  const int grid = (d.clos_n + kClosRows - 1) / kClosRows * n.parts;
  hipLaunchKernelGGL(closure_mlp_kernel, dim3(grid), dim3(64 * kClosWaves), 0, stream, d, A, n);
  HAMD_HIP(hipGetLastError());
}

}  // namespace hamd
