// Batches of independent Hilbert-form hierarchies (parameter sweeps): the
// members' host tables are packed into one set of device arrays so that one
// operator launch per Runge-Kutta stage advances every member.
#include <algorithm>
#include <array>
#include <cstdint>
#include <map>
#include <cstring>
#include <limits>
#include <string>

#include "kernels.h"
#include "qme.h"

namespace hamd {

namespace {
// workgroups that cover every item group once: a multiple of eight (the kernel
// deals consecutive eighths of the items to the eight XCDs)
int batch_groups(int n_items, int per_group, int cap) {
  const int per = (n_items + 8 * per_group - 1) / (8 * per_group);
  return std::min(8 * per, cap);
}

// a table of complex128 values in the operator precision
void upload_as(DevBuf& b, const std::vector<z128>& v, bool lo) {
  if (!lo) {
    b.upload(v);
    return;
  }
  std::vector<z64> f(v.size());
  for (size_t i = 0; i < v.size(); ++i) f[i] = conv<float>(v[i]);
  b.upload(f);
}

struct CoefRow {
  z128 iphi, psi, dir;
  int u;
};

template <typename R>
void upload_coef(DevBuf& b, const std::vector<CoefRow>& v) {
  std::vector<BatchCoef<R>> f(v.size());
  for (size_t i = 0; i < v.size(); ++i)
    f[i] = BatchCoef<R>{conv<R>(v[i].iphi), conv<R>(v[i].psi), conv<R>(v[i].dir), v[i].u, 0};
  b.upload(f);
}
}  // namespace

void Qme::set_param_batch(const std::vector<Qme*>& members) {
  if (members.empty()) throw HeomError{HEOM_ERR_ARG, "batch: no members"};
  for (size_t m = 0; m < members.size(); ++m) {
    const Qme* q = members[m];
    const std::string tag = "batch member " + std::to_string(m) + ": ";
    if (!q || !q->ready) throw HeomError{HEOM_ERR_STATE, tag + "set_param has not been called"};
    if (q->kind != HEOM_HILB) throw HeomError{HEOM_ERR_UNSUPPORTED, tag + "not heom_hilb"};
    if (!q->diag_v)
      throw HeomError{HEOM_ERR_UNSUPPORTED, tag + "coupling operators must be diagonal"};
    if (q->N > 8) throw HeomError{HEOM_ERR_UNSUPPORTED, tag + "n_level > 8"};
    if (q->dtype != dtype) throw HeomError{HEOM_ERR_ARG, tag + "dtype differs from the batch"};
    if (q->opt.device != opt.device) throw HeomError{HEOM_ERR_ARG, tag + "device differs"};
  }
  kind = kBatch;
  batch_inst.clear();
  std::vector<int> lp{0};
  std::vector<Link> bl;
  std::vector<CoefRow> bc;
  std::vector<z128> gm, Hs, tab, dt;
  std::vector<BatchItem> items;
  long long elem = 0;
  int total_ado = 0;
  int rs = 0;
  N = 0;
  for (size_t m = 0; m < members.size(); ++m) {
    const Qme& q = *members[m];
    BatchInst I{};
    I.N = q.N;
    I.N2 = q.N2;
    I.elem_base = elem;
    I.rs_off = rs;
    BatchItem W{};
    W.base = elem;
    W.N = q.N;
    W.h_off = static_cast<int>(Hs.size());
    W.tab_off = static_cast<int>(tab.size());
    W.dterm_off = static_cast<int>(dt.size());
    W.coef_off = static_cast<int>(bc.size());
    W.flags = q.real_v ? kItemRealV : 0;
    bool direct = false;
    for (const LinkFlat& f : q.flat_host) direct = direct || f.u >= q.dev.n_noise;
    if (q.dev.n_noise == 1 && !direct) W.flags |= kItemOneNoise;
    rs += q.N2;
    batch_inst.push_back(I);
    const int base_link = lp.back();
    for (int l = 0; l < q.hs.n_hrchy; ++l) lp.push_back(base_link + q.link_ptr[l + 1]);
    {
      // the member's distinct coefficient triples (compared bit for bit)
      std::map<std::array<uint64_t, 7>, int> ids;
      for (const LinkFlat& f : q.flat_host) {
        std::array<uint64_t, 7> key{};
        key[0] = static_cast<uint64_t>(f.u);
        std::memcpy(&key[1], &f.iphi, sizeof(z128));
        std::memcpy(&key[3], &f.psi, sizeof(z128));
        std::memcpy(&key[5], &f.dir, sizeof(z128));
        auto it = ids.find(key);
        if (it == ids.end()) {
          it = ids.emplace(key, static_cast<int>(ids.size())).first;
          bc.push_back(CoefRow{f.iphi, f.psi, f.dir, f.u});
        }
        bl.push_back(Link{f.nbr, it->second});
      }
    }
    gm.insert(gm.end(), q.ngamma.begin(), q.ngamma.end());
    Hs.insert(Hs.end(), q.H_host.begin(), q.H_host.end());
    tab.insert(tab.end(), q.cmac_host.begin(), q.cmac_host.end());
    dt.insert(dt.end(), q.dterm_host.begin(), q.dterm_host.end());
    const int apw = 64 / q.N2;  // ADOs per wavefront
    for (int a = 0; a < q.hs.n_hrchy; a += apw) {
      W.elem = elem + static_cast<long long>(a) * q.N2;
      W.n_ado = std::min(apw, q.hs.n_hrchy - a);
      W.g = total_ado + a;
      W.l0 = base_link + q.link_ptr[a];
      W.l1 = base_link + q.link_ptr[a + 1];
      items.push_back(W);
    }
    elem += q.main_size();
    total_ado += q.hs.n_hrchy;
    N = std::max(N, q.N);
  }
  if (elem > (1LL << 31) - 1) throw HeomError{HEOM_ERR_UNSUPPORTED, "batch: state exceeds 2^31"};
  N2 = N * N;
  batch_main_size = elem;
  batch_rs_size = rs;
  hs = Hierarchy{};
  hs.n_hrchy = total_ado;
  n_links = static_cast<long long>(bl.size());
  batch_n_coef = static_cast<long long>(bc.size());
  link_ptr = lp;
  links.clear();
  coef.clear();
  diag_v = true;
  real_v = false;
  HAMD_HIP(hipSetDevice(opt.device));
  d_link_ptr.upload(lp);
  d_blink.upload(bl);
  if (lo())
    upload_coef<float>(d_bcoef, bc);
  else
    upload_coef<double>(d_bcoef, bc);
  upload_as(d_gam, gm, lo());
  upload_as(d_H, Hs, lo());
  upload_as(d_cmac, tab, lo());
  upload_as(d_dterm, dt, lo());
  d_inst.upload(batch_inst);
  d_items.upload(items);
  dev = FormDev{};
  dev.kind = kBatch;
  dev.N = N;
  dev.N2 = N2;
  dev.n_hrchy = total_ado;
  dev.main_size = elem;
  dev.link_ptr = d_link_ptr.as<int>();
  dev.blink = d_blink.as<Link>();
  dev.b_coef = d_bcoef.p;
  dev.b_gam = d_gam.p;
  dev.b_H = d_H.p;
  dev.b_tab = d_cmac.p;
  dev.b_dterm = d_dterm.p;
  dev.diag_v = 1;
  dev.n_inst = static_cast<int>(batch_inst.size());
  dev.n_items = static_cast<int>(items.size());
  dev.inst = d_inst.as<BatchInst>();
  dev.items = d_items.as<BatchItem>();
  dev.batch_grid = batch_groups(dev.n_items, 1, kMaxGrid);
  dev.batch_ipw = 1;
  dev.batch_wpb = 1;
  ready = true;
  autotune_batch();
}

// Autotuner of the persistent batch kernel: time one pass of a Runge-Kutta
// stage of the whole batch (operator, two FP64 operands, two outputs: the
// shape of an RK4 stage) for every tile shape -- work items per wavefront step
// (1 or 2) and wavefronts per workgroup (1, 2 or 4) -- and grid size (4096 or
// 16384 persistent workgroups, or one per item group), and keep the fastest
// (one item per one-wavefront workgroup unless another shape is 3% faster).  The results do not depend on the choice beyond rounding
// (the same expression per element).
void Qme::autotune_batch() {
  const long long ms = main_size();
  const size_t eb = lo() ? sizeof(z64) : sizeof(z128);
  DevBuf a, b, y, acc, acc2;
  a.alloc(eb * ms);
  b.alloc(eb * ms);
  y.alloc(sizeof(z128) * ms);
  acc.alloc(sizeof(z128) * ms);
  acc2.alloc(sizeof(z128) * ms);
  HAMD_HIP(hipMemsetAsync(a.p, 0, eb * ms, stream));
  HAMD_HIP(hipMemsetAsync(b.p, 0, eb * ms, stream));
  HAMD_HIP(hipMemsetAsync(y.p, 0, sizeof(z128) * ms, stream));
  HAMD_HIP(hipMemsetAsync(acc.p, 0, sizeof(z128) * ms, stream));
  HAMD_HIP(hipMemsetAsync(acc2.p, 0, sizeof(z128) * ms, stream));
  // two stage passes that ping-pong their input / output and accumulator
  // buffers, as consecutive Runge-Kutta stages do
  StageArgs As[2];
  for (int p = 0; p < 2; ++p) {
    StageArgs& A = As[p];
    std::memset(&A, 0, sizeof(A));
    void* in = p ? b.p : a.p;
    void* out = p ? a.p : b.p;
    void* acc_in = p ? acc2.p : acc.p;
    void* acc_out = p ? acc.p : acc2.p;
    A.mode = MODE_STAGE;
    A.in[0] = A.in[1] = in;
    A.in_lo = lo();
    A.a_re = 1e-3;
    A.npre = 2;
    for (int c = 0; c < 2; ++c) {
      A.pre[c][0] = y.p;
      A.pre[c][1] = acc_in;
      A.dst[0][c] = out;
      A.dst[1][c] = acc_out;
    }
    A.ncombo = 2;
    A.cc[0][0] = 1.0;
    A.ck[0] = 0.5;
    A.cc[1][1] = 1.0;
    A.ck[1] = 1.0 / 6.0;
    A.dst_lo[0] = lo();
  }
  const int rb = lo() ? 4 : 8;
  hipEvent_t e0, e1;
  HAMD_HIP(hipEventCreate(&e0));
  HAMD_HIP(hipEventCreate(&e1));
  float best = std::numeric_limits<float>::max();
  int best_g = batch_groups(dev.n_items, 1, kMaxGrid), best_ipw = 1, best_wpb = 1;
  tune_log.clear();
  for (int ipw : {1, 2}) {
    for (int wpb : {1, 2, 4}) {
      // one workgroup per group of ipw * wpb items, or fewer persistent ones
      const int groups = batch_groups(dev.n_items, ipw * wpb, kMaxGrid / wpb);
      std::vector<int> cands;
      for (int g : {4096, 16384})
        if (g < groups) cands.push_back(g);
      cands.push_back(groups);
      for (int g : cands) {
        dev.batch_grid = g;
        dev.batch_ipw = ipw;
        dev.batch_wpb = wpb;
        launch_operator(dev, rb, As[0], stream);  // warm-up
        launch_operator(dev, rb, As[1], stream);
        float shape_best = std::numeric_limits<float>::max();
        for (int round = 0; round < 3; ++round) {  // best of three rounds of six passes
          HAMD_HIP(hipEventRecord(e0, stream));
          for (int r = 0; r < 6; ++r) launch_operator(dev, rb, As[r & 1], stream);
          HAMD_HIP(hipEventRecord(e1, stream));
          HAMD_HIP(hipEventSynchronize(e1));
          float ms_ = 0.f;
          HAMD_HIP(hipEventElapsedTime(&ms_, e0, e1));
          shape_best = std::min(shape_best, ms_);
        }
        tune_log.push_back(TuneEntry{ipw, wpb, g, 1e3f * shape_best / 6.0f});
        if (shape_best < best) {
          best = shape_best;
          best_g = g;
          best_ipw = ipw;
          best_wpb = wpb;
        }
      }
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  // a shape other than one item per one-wavefront workgroup must be clearly
  // faster (3%): closer timings are within what separates these passes from
  // the solver's own stages
  const int plain_g = batch_groups(dev.n_items, 1, kMaxGrid);
  for (const TuneEntry& t : tune_log) {
    if (t.ipw == 1 && t.wpb == 1 && t.grid == plain_g && 1e3f * best / 6.0f > 0.97f * t.us) {
      best_g = plain_g;
      best_ipw = 1;
      best_wpb = 1;
    }
  }
  dev.batch_grid = best_g;
  dev.batch_ipw = best_ipw;
  dev.batch_wpb = best_wpb;
}

}  // namespace hamd
