// Host side of the QME: hierarchy enumeration (hrchy_space.cc:137-231),
// heom::set_param (heom.h:57-139), the per-form set_param
// (heom_hilb.h:57-68, heom_liou.h:66-119, heom_ado.h:62-189) and the upload
// of every table to HBM.
#include "qme.h"
#include "kernels.h"
#include "mlp.h"
#include "supop.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <deque>
#include <limits>
#include <numeric>
#include <string>
#include <tuple>
#include <unordered_map>

namespace hamd {

DevBuf::~DevBuf() {
  if (p) (void)hipFree(p);
}

void DevBuf::alloc(size_t b) {
  if (p) {
    HAMD_HIP(hipFree(p));
    p = nullptr;
  }
  bytes = b;
  if (b == 0) return;
  hipError_t e = hipMalloc(&p, b);
  if (e != hipSuccess) {
    p = nullptr;
    throw HeomError{HEOM_ERR_NOMEM, "hipMalloc of " + std::to_string(b) + " bytes failed: " +
                                        hipGetErrorString(e)};
  }
}

// ---------------------------------------------------------------------------
// hierarchy
// ---------------------------------------------------------------------------
namespace {
struct KeyHash {
  size_t operator()(const std::string& s) const { return std::hash<std::string>()(s); }
};
inline std::string key_of(const int* v, int K) {
  std::string s(static_cast<size_t>(K) * 2, '\0');
  for (int k = 0; k < K; ++k) {
    s[2 * k] = static_cast<char>(v[k] & 0xff);
    s[2 * k + 1] = static_cast<char>((v[k] >> 8) & 0xff);
  }
  return s;
}
}  // namespace

Hierarchy build_hierarchy(int K, int max_depth, heom_hrchy_filter filter, void* user) {
  Hierarchy hs;
  hs.n_dim = K;
  struct Item {
    std::vector<int> idx;
    int last;
    int depth;
  };
  std::deque<Item> queue;
  queue.push_back(Item{std::vector<int>(K, 0), 0, 0});
  std::unordered_map<std::string, int, KeyHash> book;
  while (!queue.empty()) {
    Item it = std::move(queue.front());
    queue.pop_front();
    int l = hs.n_hrchy++;
    book.emplace(key_of(it.idx.data(), K), l);
    hs.n.insert(hs.n.end(), it.idx.begin(), it.idx.end());
    if (it.depth + 1 <= max_depth) {
      for (int k = it.last; k < K; ++k) {
        Item nx{it.idx, k, it.depth + 1};
        ++nx.idx[k];
        if (filter && !filter(nx.idx.data(), K, nx.depth, user)) continue;
        queue.push_back(std::move(nx));
      }
    }
  }
  const int nh = hs.n_hrchy;
  hs.ptr_p1.assign(static_cast<size_t>(nh + 1) * K, nh);
  hs.ptr_m1.assign(static_cast<size_t>(nh + 1) * K, nh);
  std::vector<int> idx(K);
  for (int l = 0; l < nh; ++l) {
    std::memcpy(idx.data(), &hs.n[static_cast<size_t>(l) * K], sizeof(int) * K);
    for (int k = 0; k < K; ++k) {
      ++idx[k];
      auto f = book.find(key_of(idx.data(), K));
      if (f != book.end()) hs.ptr_p1[static_cast<size_t>(l) * K + k] = f->second;
      idx[k] -= 2;
      if (idx[k] >= 0) {
        f = book.find(key_of(idx.data(), K));
        if (f != book.end()) hs.ptr_m1[static_cast<size_t>(l) * K + k] = f->second;
      }
      ++idx[k];
    }
  }
  return hs;
}

// ---------------------------------------------------------------------------
// QME
// ---------------------------------------------------------------------------
Qme::Qme(int kind_, int dtype_, int n_level, int max_depth_, const heom_options& opt_)
    : kind(kind_), dtype(dtype_), N(n_level), N2(n_level * n_level), max_depth(max_depth_),
      opt(opt_) {
  H.assign(N2, z128{0.0, 0.0});
  HAMD_HIP(hipSetDevice(opt.device));
  HAMD_HIP(hipStreamCreate(&stream));
}

Qme::~Qme() {
  if (stream) (void)hipStreamDestroy(stream);
}

using namespace supop;

// Every change of the operator begins here (set_param, binding, unbinding).
void Qme::clear_closure() {
  ++generation;
  closure.reset();
  dev.clos = nullptr;
  dev.clos_lo = dev.clos_n = 0;
}

StageArgs Qme::diff_args(void* drho, const void* rho, z128 alpha, z128 beta) const {
  const int l = lo() ? 1 : 0;
  StageArgs A;
  std::memset(&A, 0, sizeof(A));
  A.mode = MODE_DIFF;
  A.in[0] = A.in[1] = rho;
  A.in_lo = l;
  A.dst[0][0] = A.dst[0][1] = drho;
  A.dst_lo[0] = l;
  if (beta.re != 0.0 || beta.im != 0.0) {
    A.npre = 1;
    A.pre[0][0] = A.pre[1][0] = drho;
    A.pre_lo = l ? 1u : 0u;
  }
  A.a_re = alpha.re;
  A.a_im = alpha.im;
  A.b_re = beta.re;
  A.b_im = beta.im;
  return A;
}

int Qme::operate(int real_bytes, const StageArgs& A, hipStream_t st) {
  if (closure) closure->forward(*this, A, st);
  return launch_operator(dev, real_bytes, A, st);
}

void Qme::set_param() {
  clear_closure();
  const int nn = static_cast<int>(noise.size());
  if (!H_set) throw HeomError{HEOM_ERR_ARG, "set_param: H not set"};
  if (nn == 0) throw HeomError{HEOM_ERR_ARG, "set_param: alloc_noises not called"};
  for (int u = 0; u < nn; ++u)
    if (!noise[u].set)
      throw HeomError{HEOM_ERR_ARG, "set_param: noise " + std::to_string(u) + " not set"};
  uploaded = false;
  if (redfield()) {
    set_param_redfield();
    uploaded = true;
    return;
  }

  // col_major storage is the transposed row-major problem with
  // H -> -H^T, V -> -V^T, A -> -A, gamma -> gamma^T (heom_hilb.h:148-162).
  std::vector<z128> Hw = H;
  std::vector<NoiseParams> nz = noise;
  if (opt.order == 1) {
    for (int i = 0; i < N; ++i)
      for (int j = 0; j < N; ++j) Hw[i * N + j] = zscale(-1.0, H[j * N + i]);
    for (auto& z : nz) {
      std::vector<z128> V2(N2);
      for (int i = 0; i < N; ++i)
        for (int j = 0; j < N; ++j) V2[i * N + j] = zscale(-1.0, z.V[j * N + i]);
      z.V = V2;
      for (auto& x : z.A) x = zscale(-1.0, x);
      std::vector<z128> g2(z.gamma.size());
      for (int i = 0; i < z.len; ++i)
        for (int j = 0; j < z.len; ++j) g2[i * z.len + j] = z.gamma[j * z.len + i];
      z.gamma = g2;
    }
  }

  // heom::set_param: lk linearisation (heom.h:66-74)
  lk.assign(nn, {});
  int K = 0;
  for (int u = 0; u < nn; ++u)
    for (int k = 0; k < nz[u].len; ++k) lk[u].push_back(K++);
  if (K == 0) throw HeomError{HEOM_ERR_ARG, "set_param: no bath modes"};
  if (max_depth < 0) throw HeomError{HEOM_ERR_ARG, "set_param: max_depth < 0"};

  hs = build_hierarchy(K, max_depth, hrchy_filter, hrchy_filter_user);
  const int nh = hs.n_hrchy;
  if (static_cast<long long>(nh) * N2 > (1LL << 31) - 1)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "set_param: main_size exceeds 2^31"};

  // Gamma_n (heom.h:93-104)
  ngamma.assign(nh, z128{0.0, 0.0});
  for (int l = 0; l < nh; ++l) {
    z128 g{0.0, 0.0};
    for (int u = 0; u < nn; ++u)
      for (int k = 0; k < nz[u].len; ++k)
        g = g + zscale(static_cast<double>(hs.n[static_cast<size_t>(l) * K + lk[u][k]]),
                       nz[u].gamma[k * nz[u].len + k]);
    ngamma[l] = g;
  }

  // s = S phi_0, a = A phi_0 (heom.h:123-138)
  s.assign(nn, {});
  a.assign(nn, {});
  for (int u = 0; u < nn; ++u) {
    const int len = nz[u].len;
    s[u].assign(len, z128{0.0, 0.0});
    a[u].assign(len, z128{0.0, 0.0});
    for (int i = 0; i < len; ++i)
      for (int j = 0; j < len; ++j) {
        s[u][i] = s[u][i] + zmul(nz[u].S[i * len + j], nz[u].phi0[j]);
        a[u][i] = a[u][i] + zmul(nz[u].A[i * len + j], nz[u].phi0[j]);
      }
  }

  diag_v = true;
  for (int u = 0; u < nn && diag_v; ++u)
    for (int i = 0; i < N && diag_v; ++i)
      for (int j = 0; j < N; ++j)
        if (i != j && !zzero(nz[u].V[i * N + j])) {
          diag_v = false;
          break;
        }

  real_v = diag_v;
  for (int u = 0; u < nn && real_v; ++u)
    for (int i = 0; i < N; ++i)
      if (nz[u].V[i * N + i].im != 0.0) {
        real_v = false;
        break;
      }

  noise_work_ = nz;
  H_work_ = Hw;
  build_links();

  if ((kind == HEOM_LIOU || kind == HEOM_ADO) && N > 32)
    throw HeomError{HEOM_ERR_UNSUPPORTED, "heom_liou/heom_ado: n_level > 32"};
  upload();
  uploaded = true;
  ready = true;
}

void Qme::build_links() {
  const int nn = static_cast<int>(noise_work_.size());
  const int K = hs.n_dim, nh = hs.n_hrchy, pv = nh;
  const bool sq = opt.sqrt_norm != 0;
  // coefficient dedup: (type, mode, n_j, n_k, j, k) -> cid
  std::map<std::tuple<int, int, int, int, int, int>, int> cmap;
  coef.clear();
  auto get = [&](std::tuple<int, int, int, int, int, int> key, const Coef& c) {
    auto f = cmap.find(key);
    if (f != cmap.end()) return f->second;
    int id = static_cast<int>(coef.size());
    coef.push_back(c);
    cmap.emplace(key, id);
    return id;
  };
  link_ptr.assign(nh + 1, 0);
  links.clear();
  for (int l = 0; l < nh; ++l) {
    const int* nl = &hs.n[static_cast<size_t>(l) * K];
    for (int u = 0; u < nn; ++u) {
      const NoiseParams& z = noise_work_[u];
      // +1 terms (heom_hilb.h:170-182)
      for (int k = 0; k < z.len; ++k) {
        int mode = lk[u][k];
        int p = hs.ptr_p1[static_cast<size_t>(l) * K + mode];
        if (p == pv) continue;
        int nk = nl[mode];
        Coef c{};
        c.phi = sq ? zscale(std::sqrt(nk + 1.0), z.sigma[k]) : z.sigma[k];
        c.u = u;
        links.push_back(Link{p, get(std::make_tuple(0, mode, 0, sq ? nk : 0, 0, 0), c)});
      }
      // -1 terms (heom_hilb.h:184-198)
      for (int k = 0; k < z.len; ++k) {
        int mode = lk[u][k];
        int m = hs.ptr_m1[static_cast<size_t>(l) * K + mode];
        if (m == pv) continue;
        int nk = nl[mode];
        double f = sq ? std::sqrt(static_cast<double>(nk)) : static_cast<double>(nk);
        Coef c{};
        c.phi = zscale(f, s[u][k]);
        c.psi = zscale(-f, a[u][k]);
        c.u = u;
        links.push_back(Link{m, get(std::make_tuple(1, mode, 0, nk, 0, 0), c)});
      }
    }
    // off-diagonal gamma (heom_hilb.h:128-147); dropped in parity mode
    if (!opt.parity_q1) {
      for (int u = 0; u < nn; ++u) {
        const NoiseParams& z = noise_work_[u];
        for (int j = 0; j < z.len; ++j)
          for (int k = 0; k < z.len; ++k) {
            z128 v = z.gamma[j * z.len + k];
            if (j == k || zzero(v)) continue;
            int mj = lk[u][j], mk = lk[u][k];
            int q1 = hs.ptr_m1[static_cast<size_t>(l) * K + mj];
            if (q1 == pv) continue;
            int q = hs.ptr_p1[static_cast<size_t>(q1) * K + mk];
            if (q == pv) continue;
            int nj = nl[mj], nk = nl[mk];
            double f = sq ? std::sqrt(nj * (nk + 1.0)) : static_cast<double>(nj);
            Coef c{};
            c.dir = zscale(f, v);
            c.u = nn;
            links.push_back(Link{q, get(std::make_tuple(2, u, nj, nk, j, k), c)});
          }
      }
    }
    link_ptr[l + 1] = static_cast<int>(links.size());
  }
}

// Workgroups are dealt to the eight XCDs round-robin, and the neighbours an
// ADO reads are cheap only when they sit in the same XCD's L2.  ADOs are
// therefore listed in depth-first preorder of the tree in which every ADO hangs
// from the one that generated it in the breadth-first enumeration (n - e_k, k
// its highest occupied mode: hrchy_space.cc:160-198 pushes n + e_k only for k
// at or above the mode last raised), cut into eight consecutive parts of equal
// size (the ADOs and their links then mix the tiers evenly), and each part is
// given back in breadth-first order to workgroups x, x + 8, x + 16, ...
// Subtrees stay together, so most +-1 links join ADOs of one part.
std::vector<BlockMap> Qme::build_block_map() const {
  const int nh = hs.n_hrchy, K = hs.n_dim;
  constexpr int P = 8;
  std::vector<int> order;
  order.reserve(nh);
  std::vector<char> seen(nh, 0);
  std::vector<int> stack{0};
  while (!stack.empty()) {
    const int g = stack.back();
    stack.pop_back();
    if (g < 0 || g >= nh || seen[g]) continue;
    seen[g] = 1;
    order.push_back(g);
    const int* ng = &hs.n[static_cast<size_t>(g) * K];
    int top = 0;
    for (int k = 0; k < K; ++k)
      if (ng[k] > 0) top = k;
    for (int k = K - 1; k >= top; --k) {  // lower modes are visited first
      const int c = hs.ptr_p1[static_cast<size_t>(g) * K + k];
      if (c != nh) stack.push_back(c);
    }
  }
  for (int g = 0; g < nh; ++g)  // anything the tree walk missed keeps its order
    if (!seen[g]) order.push_back(g);
  std::vector<std::vector<int>> part(P);
  size_t pos = 0;
  for (int x = 0; x < P; ++x) {
    const int cnt = (nh - x + P - 1) / P;  // workgroups b < nh with b % 8 == x
    part[x].assign(order.begin() + pos, order.begin() + pos + cnt);
    std::sort(part[x].begin(), part[x].end());
    pos += cnt;
  }
  std::vector<BlockMap> map(nh);
  for (int x = 0; x < P; ++x)
    for (size_t i = 0; i < part[x].size(); ++i) {
      const int g = part[x][i];
      map[i * P + x] = BlockMap{g, link_ptr[g], link_ptr[g + 1], 0};
    }
  return map;
}

// Work units of hilb_split_kernel, from the work-unit map: unit b keeps to XCD
// b mod 8, whose ADOs stay the ones of the map.  An ADO with more links than a
// quarter (a half, N > 11) of the most any has is shared by a unit's groups, the
// others fill units together, in the map's order.
// Used while the ADOs are at most 4096 wavefronts (2048 with two groups) and some
// ADO has more links than the one-group kernels take in two rounds.  RK4 stages
// with launch, one group -> shared: 253 ADOs of 7x7 9.8 -> 5.6 us, 1820 of 4x4
// 8.2 -> 5.6, 1771 of 10x10 (3542 wavefronts) 10.9 -> 9.8, 325 of 12x12 11.3 -> 8.7;
// past the line the chip is full, and the shared kernel's registers and
// workgroups cost more than its shorter chain: 4060 of 9x9 13.7 -> 18.3,
// 969 of 16x16 11.1 -> 12.3, 12 650 of 7x7 17.4 -> 24.4.
void Qme::build_split_units(const std::vector<BlockMap>& bm) {
  dev.sunits = nullptr;
  dev.slinks = nullptr;
  dev.n_sunits = dev.slink_n = 0;
  int most = 0;
  for (const BlockMap& b : bm) most = std::max(most, b.l1 - b.l0);
  const long long waves = static_cast<long long>(hs.n_hrchy) * ((N2 + 63) / 64);
  const int G = split_groups(N);
  if (dev.kind != HEOM_HILB || !dev.diag_v || N < 4 || N > 16 || most <= 8 ||
      waves > 1024 * G || split_vd_lds(dev.n_noise, N, false, sizeof(double)) > 32 * 1024)
    return;
  constexpr int P = 8;
  const int per = (most + G - 1) / G;
  struct Group {
    int g, l0, l1, step, shared;  // links l0, l0 + step, ... below l1
  };
  std::vector<Group> x[P];
  for (int p = 0; p < P; ++p) {
    std::vector<Group> few;
    for (size_t b = p; b < bm.size(); b += P) {
      if (bm[b].l1 - bm[b].l0 > per)
        for (int q = 0; q < G; ++q) x[p].push_back({bm[b].g, bm[b].l0 + q, bm[b].l1, G, 1});
      else
        few.push_back({bm[b].g, bm[b].l0, bm[b].l1, 1, 0});
    }
    while (few.size() % G) few.push_back({-1, 0, 0, 1, 0});
    x[p].insert(x[p].end(), few.begin(), few.end());
  }
  size_t n = 0;  // groups per XCD
  for (auto& v : x) n = std::max(n, v.size());
  std::vector<SplitUnit> units(n * P, SplitUnit{-1, 0});
  std::vector<Link> slots(n * P * per, Link{-1, 0});
  for (int p = 0; p < P; ++p)
    for (size_t y = 0; y < x[p].size(); ++y) {
      const Group& gr = x[p][y];
      const size_t at = (y / G * P + p) * G + y % G;
      units[at] = SplitUnit{gr.g, gr.shared};
      size_t t = at * per;
      for (int l = gr.l0; l < gr.l1; l += gr.step) slots[t++] = links[l];
    }
  // one buffer for both: an allocation and a copy are 25 us each of the set-up
  std::vector<char> all(sizeof(SplitUnit) * units.size() + sizeof(Link) * slots.size());
  static_assert(sizeof(SplitUnit) % alignof(Link) == 0, "slots follow the units");
  std::memcpy(all.data(), units.data(), sizeof(SplitUnit) * units.size());
  std::memcpy(all.data() + sizeof(SplitUnit) * units.size(), slots.data(),
              sizeof(Link) * slots.size());
  d_sunits.upload(all);
  dev.sunits = d_sunits.as<SplitUnit>();
  dev.slinks = reinterpret_cast<const Link*>(d_sunits.as<SplitUnit>() + units.size());
  dev.n_sunits = static_cast<int>(n * P / G);
  dev.slink_n = per;
}

void Qme::upload() {
  const int nn = static_cast<int>(noise_work_.size());
  HAMD_HIP(hipSetDevice(opt.device));
  d_link_ptr.upload(link_ptr);
  d_links.upload(links);
  const std::vector<BlockMap> bm = build_block_map();
  d_bmap.upload(bm);
  std::vector<LinkFlat> flat(links.size());
  for (size_t l = 0; l < links.size(); ++l) {
    const Coef& cf = coef[links[l].cid];
    LinkFlat f{};
    f.nbr = links[l].nbr;
    f.u = cf.u;
    f.iphi = z128{-cf.phi.im, cf.phi.re};  // i*phi
    f.psi = cf.psi;
    f.dir = cf.dir;
    flat[l] = f;
  }
  d_flat.upload(flat);
  flat_host = flat;
  n_links = static_cast<long long>(links.size());
  {
    // (v_i - v_j, v_i + v_j) per noise and element, one zero row for direct links
    std::vector<z128> tab;
    if (diag_v) {
      const size_t rows = static_cast<size_t>(nn + 1) * N2;
      tab.assign(real_v ? rows : 2 * rows, z128{0.0, 0.0});
      for (int u = 0; u < nn; ++u)
        for (int i = 0; i < N; ++i)
          for (int j = 0; j < N; ++j) {
            const z128 vi = noise_work_[u].V[i * N + i], vj = noise_work_[u].V[j * N + j];
            const size_t b = static_cast<size_t>(u) * N2 + i * N + j;
            if (real_v) {
              tab[b] = z128{vi.re - vj.re, vi.re + vj.re};
            } else {
              tab[2 * b] = vi - vj;
              tab[2 * b + 1] = vi + vj;
            }
          }
    }
    d_cmac.upload(tab);
    cmac_host = tab;
  }
  d_coef.upload(coef);
  d_gam.upload(ngamma);
  d_H.upload(H_work_);
  std::vector<z128> V(static_cast<size_t>(nn) * N2), Vd(static_cast<size_t>(nn) * N),
      sd(nn), dterm(N2, z128{0.0, 0.0});
  for (int u = 0; u < nn; ++u) {
    std::copy(noise_work_[u].V.begin(), noise_work_[u].V.end(), V.begin() + u * N2);
    for (int i = 0; i < N; ++i) Vd[u * N + i] = noise_work_[u].V[i * N + i];
    sd[u] = noise_work_[u].s_delta;
  }
  if (diag_v) {
    for (int i = 0; i < N; ++i)
      for (int j = 0; j < N; ++j) {
        z128 acc{0.0, 0.0};
        for (int u = 0; u < nn; ++u) {
          z128 c = Vd[u * N + i] - Vd[u * N + j];
          acc = acc + zmul(noise_work_[u].s_delta, zmul(c, c));
        }
        dterm[i * N + j] = acc;
      }
  }
  d_V.upload(V);
  d_Vd.upload(Vd);
  d_dterm.upload(dterm);
  dterm_host = dterm;
  H_host = H_work_;
  d_sdelta.upload(sd);
  // heom_liou and heom_ado (heom_liou.h:151-255, heom_ado.h:191-202) apply the
  // same operator as superoperators of up to N^4 entries (per ADO, or merged over
  // the hierarchy): a commutator or an anticommutator from the left and the right
  // is 2 N products per element where the sparse row is 2 N - 1 gathered ones, so
  // the Hilbert-form kernels compute all three forms.  (160 stages on the 7-site
  // chain at depth 2: 4.3 ms with per-ADO sparse rows, 1.7 ms here.)
  const bool hilb = kind == HEOM_HILB || kind == HEOM_LIOU || kind == HEOM_ADO;
  bool diag = diag_v;
  // those two forms take any number of noises: past the LDS tables of the diagonal
  // kernels (see launch_hilb_n) they use the dense one
  if (hilb && kind != HEOM_HILB && N <= 16 &&
      sizeof(z128) * (nn + 1) * static_cast<size_t>(N) > 48 * 1024)
    diag = false;
  dev.kind = hilb ? HEOM_HILB : kind;
  dev.N = N;
  dev.N2 = N2;
  dev.n_hrchy = hs.n_hrchy;
  dev.n_noise = nn;
  dev.main_size = main_size();
  dev.link_ptr = d_link_ptr.as<int>();
  dev.links = d_links.as<Link>();
  dev.coef = d_coef.as<Coef>();
  dev.gam = d_gam.as<z128>();
  dev.H = d_H.as<z128>();
  dev.V = d_V.as<z128>();
  dev.Vd = d_Vd.as<z128>();
  dev.dterm = d_dterm.as<z128>();
  dev.sdelta = d_sdelta.as<z128>();
  dev.diag_v = diag ? 1 : 0;
  dev.real_v = real_v ? 1 : 0;
  dev.flat = d_flat.as<LinkFlat>();
  dev.bmap = d_bmap.as<BlockMap>();
  build_split_units(bm);
  dev.cmac_tab = d_cmac.as<z128>();
  dev.max_links = 0;
  for (int l = 0; l < hs.n_hrchy; ++l)
    dev.max_links = std::max(dev.max_links, link_ptr[l + 1] - link_ptr[l]);
  // matrix-core commutator: heom_hilb, 16 < N <= 64, diagonal V (tiles of 32, 48
  // or 64 rows; H is zero-padded to the tile in its planes)
  const bool big = hilb && N > 16 && N <= 64;
  const bool mfma_ok = big && diag_v;
  const bool mfma_dense = big && !diag_v;
  dev.mfma = 0;
  dev.tile = mfma_tile(N, mfma_dense, lo());
  if (opt.matrix_cores && mfma_ok) dev.mfma = dtype == HEOM_C64_BF16X3 ? 2 : 1;
  if (opt.matrix_cores && mfma_dense && dtype != HEOM_C64_BF16X3) dev.mfma = 3;
  if (kind != HEOM_HILB) {
    // heom_liou / heom_ado: matrix_cores = 0 has no vector kernel for dense V, and
    // many noises leave the LDS tables of the matrix-core kernel
    if (mfma_dense) dev.mfma = 3;
    if (mfma_ok && 2 * sizeof(double) * 32 * 33 + sizeof(z128) * (nn + 1) * static_cast<size_t>(N) >
                       kMfmaLdsCap)
      dev.mfma = 0;
  }
  if (dtype == HEOM_C64_BF16X3 && (dev.mfma != 2 || kind != HEOM_HILB))
    throw HeomError{HEOM_ERR_UNSUPPORTED,
                    "HEOM_C64_BF16X3 is provided for heom_hilb with 16 < n_level <= 64, diagonal "
                    "coupling operators and matrix_cores = 1"};
  dev.real_h = 1;
  {
    // real / imaginary planes of H with leading dimension P (the MFMA tile,
    // zero-padded), P = N outside the matrix-core path
    const int P = (mfma_ok || mfma_dense) ? dev.tile : N;
    std::vector<double> hr(static_cast<size_t>(P) * P, 0.0), hi(hr.size(), 0.0);
    std::vector<float> hr32(hr.size(), 0.f), hi32(hr.size(), 0.f);
    for (int i = 0; i < N; ++i)
      for (int j = 0; j < N; ++j) {
        const z128 h = H_work_[i * N + j];
        const size_t e = static_cast<size_t>(i) * P + j;
        hr[e] = h.re;
        hi[e] = h.im;
        hr32[e] = static_cast<float>(h.re);
        hi32[e] = static_cast<float>(h.im);
        if (h.im != 0.0) dev.real_h = 0;
      }
    d_Hre.upload(hr);
    d_Him.upload(hi);
    d_Hre32.upload(hr32);
    d_Him32.upload(hi32);
  }
  dev.real_vd = 1;
  if (dev.mfma == 3) {
    // every V_u zero-padded to the tile, as real / imaginary planes
    const int P = dev.tile;
    const size_t pl = static_cast<size_t>(P) * P;
    std::vector<double> vr(pl * nn, 0.0), vi(vr.size(), 0.0);
    std::vector<float> vr32(vr.size(), 0.f), vi32(vr.size(), 0.f);
    for (int u = 0; u < nn; ++u)
      for (int i = 0; i < N; ++i)
        for (int j = 0; j < N; ++j) {
          const z128 v = noise_work_[u].V[i * N + j];
          const size_t e = u * pl + static_cast<size_t>(i) * P + j;
          vr[e] = v.re;
          vi[e] = v.im;
          vr32[e] = static_cast<float>(v.re);
          vi32[e] = static_cast<float>(v.im);
          if (v.im != 0.0) dev.real_vd = 0;
        }
    d_Vre.upload(vr);
    d_Vim.upload(vi);
    d_Vre32.upload(vr32);
    d_Vim32.upload(vi32);
  }
  dev.Vre = d_Vre.as<double>();
  dev.Vim = d_Vim.as<double>();
  dev.Vre32 = d_Vre32.as<float>();
  dev.Vim32 = d_Vim32.as<float>();
  dev.Hre = d_Hre.as<double>();
  dev.Him = d_Him.as<double>();
  dev.Hre32 = d_Hre32.as<float>();
  dev.Him32 = d_Him32.as<float>();
}

}  // namespace hamd
