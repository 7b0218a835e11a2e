// RK4 (rk4.h:40-65) and Dormand-Prince 5(4) (rkdp.h:21-179) drivers.  Every
// stage is one fused operator pass (kernels.hip).  The Dormand-Prince step
// control and the walk through the output times run on the device; the host
// keeps one attempt queued behind the running one and reads a progress word in
// host memory instead of synchronising.
#include "solver.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <set>
#include <thread>

#include "kernels.h"

namespace hamd {

namespace {
// slot numbers
enum {
  SL_Y = 0, SL_YNEW = 1, SL_Y32 = 2, SL_YNEW32 = 3,
  SL_SA = 4, SL_SB = 5, SL_ACC = 6, SL_K1 = 7,  // K2..K5 = 8..11
  SL_E = 13,  // Dormand-Prince: sum_{j<6} E_j k_j, always FP64
  // Dormand-Prince: D of y and of y_new (k_1 = -dt*D(y) for any dt: an attempt's last
  // evaluation is the next attempt's first, and a rejected attempt keeps its own)
  SL_D = 14, SL_DNEW = 15
};
}  // namespace

int StageSpec::pre_index(int slot) {
  for (size_t s = 0; s < pre.size(); ++s)
    if (pre[s] == slot) return static_cast<int>(s);
  if (static_cast<int>(pre.size()) >= kMaxPre)
    throw HeomError{HEOM_ERR_STATE, "stage needs too many operands"};
  pre.push_back(slot);
  return static_cast<int>(pre.size()) - 1;
}

// dst (dst2) <- sum of terms (in the given order) + ckv*k
void StageSpec::combo(const std::vector<std::pair<int, double>>& terms, double ckv, int d,
                      int d2) {
  const int c = ncombo++;
  int last = -1;
  for (auto& t : terms) {
    const int s = pre_index(t.first);
    if (s <= last) throw HeomError{HEOM_ERR_STATE, "combination order differs from operands"};
    last = s;
    cc[c][s] = t.second;
  }
  ck[c] = ckv;
  dst[c] = d;
  dst2[c] = d2;
}

Solver::Solver(std::shared_ptr<Qme> q_, int kind_)
    : q_owner(std::move(q_)), q(q_owner.get()), kind(kind_) {
  if (!q) throw HeomError{HEOM_ERR_ARG, "solver: null QME"};
  if (!q->ready) throw HeomError{HEOM_ERR_STATE, "solver: set_param has not been called"};
  if (kind != HEOM_RK4 && kind != HEOM_RKDP && kind != HEOM_LSRK4)
    throw HeomError{HEOM_ERR_ARG, "solver: unknown solver kind"};
  HAMD_HIP(hipSetDevice(q->opt.device));
  in_bytes = q->lo() ? 4 : 8;
  ms = q->main_size();
  const size_t z128b = sizeof(z128) * ms;
  const size_t sinb = (in_bytes == 4 ? sizeof(z64) : sizeof(z128)) * ms;
  const int lo = in_bytes == 4 ? 1 : 0;
  auto mk = [&](int s, size_t b, int is_lo) {
    P[s].alloc(b);
    HAMD_HIP(hipMemset(P[s].p, 0, b));
    sp[s] = P[s].p;
    slo[s] = is_lo;
  };
  mk(SL_Y, z128b, 0);
  // Dormand-Prince: the y / y_new pair; lsrk4: the state alternates between them
  if (kind != HEOM_RK4) mk(SL_YNEW, z128b, 0);
  if (lo) {
    mk(SL_Y32, sinb, 1);
    if (kind != HEOM_RK4) mk(SL_YNEW32, sinb, 1);
  }
  if (kind != HEOM_LSRK4) {
    mk(SL_SA, sinb, lo);
    mk(SL_SB, sinb, lo);
  }
  if (kind == HEOM_RK4 || kind == HEOM_LSRK4) {
    mk(SL_ACC, z128b, 0);  // rk4: the accumulator; lsrk4: buff
  } else {
    // the error sum takes the buffer of k_2, which no stage reads any more when it is
    // written (B_2 = E_2 = 0): ten state blocks (complex64: 7.5) in all
    mk(SL_K1 + 1, z128b, lo);
    sp[SL_E] = P[SL_K1 + 1].p;
    for (int k = 2; k < 5; ++k) mk(SL_K1 + k, sinb, lo);
    mk(SL_D, sinb, lo);
    mk(SL_DNEW, sinb, lo);
  }
  if (q->opt.renorm_rho0) {
    if (q->kind == kBatch)
      throw HeomError{HEOM_ERR_UNSUPPORTED, "renorm_rho0 is not provided for batches"};
    if (q->N > 64) throw HeomError{HEOM_ERR_UNSUPPORTED, "renorm_rho0: n_level > 64"};
    d_tr0.alloc(sizeof(double));
  }
  d_ctrl.alloc(2 * sizeof(Ctrl));
  HAMD_HIP(hipMemset(d_ctrl.p, 0, 2 * sizeof(Ctrl)));
  d_partials.alloc(sizeof(double) * kMaxGrid);
  HAMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&h_ctrl), sizeof(Ctrl) + 128,
                         hipHostMallocCoherent));
  std::memset(h_ctrl, 0, sizeof(Ctrl));
  // the progress word on a cache line of its own
  const uintptr_t after = reinterpret_cast<uintptr_t>(h_ctrl) + sizeof(Ctrl);
  mail = reinterpret_cast<unsigned long long*>((after + 63) & ~uintptr_t(63));
  build_stages(0.0, 0.0);
}

Solver::~Solver() {
  graphs.clear();
  if (rec_stream) (void)hipStreamDestroy(rec_stream);
  if (h_ctrl) (void)hipHostFree(h_ctrl);
  if (h_times) (void)hipHostFree(h_times);
  if (h_state) (void)hipHostFree(h_state);
}

// Output times to device memory by way of pinned memory: no allocation, and no
// wait, while the list is no longer than an earlier one.  Both buffers are idle:
// every solve waits for its stream before it returns.
void Solver::upload_times(const double* t, int n) {
  if (n > n_times) {
    if (h_times) (void)hipHostFree(h_times);
    h_times = nullptr;
    n_times = 0;
    HAMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&h_times), sizeof(double) * n,
                           hipHostMallocDefault));
    d_res_t.alloc(sizeof(double) * n);
    n_times = n;
  }
  std::memcpy(h_times, t, sizeof(double) * n);
  HAMD_HIP(hipMemcpyAsync(d_res_t.p, h_times, sizeof(double) * n, hipMemcpyHostToDevice,
                          q->stream));
}

// A small list to a device buffer that is kept while the lists fit (idle, as above)
void Solver::upload_kept(DevBuf& b, const void* src, size_t bytes) {
  if (b.bytes < bytes) b.alloc(bytes);
  HAMD_HIP(hipMemcpyAsync(b.p, src, bytes, hipMemcpyHostToDevice, q->stream));
}

// Workspace of a solve call (its state or rho_S in device memory): kept up to
// kKeepWork bytes, so that repeated solves allocate nothing; a larger one is the
// call's own.
void* Solver::workspace(DevBuf& kept, DevBuf& own, size_t bytes) {
  if (bytes > kKeepWork) {
    own.alloc(bytes);
    return own.p;
  }
  if (kept.bytes < bytes) kept.alloc(bytes);
  return kept.p;
}

void Solver::check_qme() const {
  if (!q->ready)
    throw HeomError{HEOM_ERR_STATE, "solver: the QME's parameters changed and set_param has not "
                                    "been called again"};
  if (q->main_size() != ms)
    throw HeomError{HEOM_ERR_STATE, "solver: the QME's main_size changed since the solver was "
                                    "created; create a new solver"};
}

bool Solver::operator_changed(unsigned long long& gen) {
  if (q->generation == gen) return false;
  gen = q->generation;
  graphs.clear();
  graph_warm = false;
  if (!q->uploaded || q->main_size() != ms)
    throw HeomError{HEOM_ERR_STATE, "solver: set_param failed or changed the main_size during a "
                                    "solve"};
  return true;
}

// Physical buffer of a slot for ping-pong parity `cur` (slots 0..3 and the D
// pair swap within their pair when cur == 1).
void* Solver::slot_ptr(int s, int cur) const {
  if (s < 0) return nullptr;
  if (s < 4 || s >= SL_D) return sp[s ^ cur];
  return sp[s];
}

StageArgs Solver::resolve(const StageSpec& s) const {
  StageArgs a;
  std::memset(&a, 0, sizeof(a));
  a.mode = MODE_STAGE;
  const bool pp = kind == HEOM_RKDP;  // ping-pong pairs only with the control block
  for (int cur = 0; cur < 2; ++cur) {
    const int c = pp ? cur : 0;
    a.in[cur] = slot_ptr(s.in_slot, c);
    a.k[cur] = slot_ptr(s.k_slot, c);
    for (size_t j = 0; j < s.pre.size(); ++j) a.pre[cur][j] = slot_ptr(s.pre[j], c);
    for (int k = 0; k < 2; ++k) {
      a.dst[k][cur] = slot_ptr(s.dst[k], c);
      a.dst2[k][cur] = slot_ptr(s.dst2[k], c);
    }
  }
  a.in_lo = slo[s.in_slot];
  a.npre = static_cast<int>(s.pre.size());
  for (size_t j = 0; j < s.pre.size(); ++j)
    if (s.pre[j] >= 0 && slo[s.pre[j]]) a.pre_lo |= 1u << j;
  a.k_lo = s.k_slot >= 0 ? slo[s.k_slot] : 0;
  a.epi = kind != HEOM_RKDP ? EPI_RK : s.k_slot >= SL_D ? EPI_D : EPI_K;
  if (a.epi == EPI_K && (s.pre.size() < 2 || s.pre[1] != SL_D))
    throw HeomError{HEOM_ERR_STATE, "Dormand-Prince stage without D as operand 1"};
  a.ncombo = s.ncombo;
  std::memcpy(a.cc, s.cc, sizeof(a.cc));
  std::memcpy(a.ck, s.ck, sizeof(a.ck));
  for (int k = 0; k < 2; ++k) {
    a.dst_lo[k] = s.dst[k] >= 0 ? slo[s.dst[k]] : 0;
    a.dst2_lo[k] = s.dst2[k] >= 0 ? slo[s.dst2[k]] : 0;
  }
  a.do_err = s.do_err;
  a.ek = s.ek;
  if (kind == HEOM_RKDP) a.ctrl = ctrl_dev();
  a.partials = partials_dev();
  return a;
}

void Solver::build_stages(double atol, double rtol) {
  specs.clear();
  stages.clear();
  graphs.clear();
  graph_warm = false;
  direct_attempts = 0;
  const bool lo = in_bytes == 4;
  const int y_in = lo ? SL_Y32 : SL_Y;
  if (kind == HEOM_RK4) {
    // rk4.h:47-64; k2 and k3 enter the accumulator as soon as they exist
    StageSpec a;
    a.in_slot = y_in;
    a.combo({{SL_Y, 1.0}}, 0.5, SL_SA);
    a.combo({{SL_Y, 1.0}}, 1.0 / 6.0, SL_ACC);
    specs.push_back(a);

    a = StageSpec();
    a.in_slot = SL_SA;
    a.combo({{SL_Y, 1.0}}, 0.5, SL_SB);
    a.combo({{SL_ACC, 1.0}}, 2.0 / 6.0, SL_ACC);
    specs.push_back(a);

    a = StageSpec();
    a.in_slot = SL_SB;
    a.combo({{SL_Y, 1.0}}, 1.0, SL_SA);
    a.combo({{SL_ACC, 1.0}}, 2.0 / 6.0, SL_ACC);
    specs.push_back(a);

    a = StageSpec();
    a.in_slot = SL_SA;
    a.combo({{SL_ACC, 1.0}}, 1.0 / 6.0, SL_Y, lo ? SL_Y32 : -1);
    specs.push_back(a);
  } else if (kind == HEOM_LSRK4) {
    // lsrk4.h:33-48: buff = beta*buff + k (k = -dt*D) with beta = 0, -1, -1, -1,
    // then rho += c*buff, c = 1/3, 3/4, 2/3, 1/4.  The state alternates between
    // y and y_new (neighbour reads never see a half-written state); rho + c*buff
    // is formed as rho + c*beta*buff + c*k from the operands before the update.
    const double beta[4] = {0.0, -1.0, -1.0, -1.0};
    const double c[4] = {1.0 / 3.0, 3.0 / 4.0, 2.0 / 3.0, 1.0 / 4.0};
    const int src[4] = {SL_Y, SL_YNEW, SL_Y, SL_YNEW};
    const int dst[4] = {SL_YNEW, SL_Y, SL_YNEW, SL_Y};
    const int src32[4] = {SL_Y32, SL_YNEW32, SL_Y32, SL_YNEW32};
    for (int s = 0; s < 4; ++s) {
      StageSpec a;
      a.in_slot = lo ? src32[s] : src[s];
      if (beta[s] == 0.0) {
        a.combo({{src[s], 1.0}}, c[s], dst[s], lo ? src32[(s + 1) % 4] : -1);
        a.combo({}, 1.0, SL_ACC);
      } else {
        a.combo({{src[s], 1.0}, {SL_ACC, c[s] * beta[s]}}, c[s], dst[s],
                lo ? src32[(s + 1) % 4] : -1);
        a.combo({{SL_ACC, beta[s]}}, 1.0, SL_ACC);
      }
      specs.push_back(a);
    }
  } else {
    // Dormand-Prince: stage 0 evaluates D(y), stores it and forms the input of stage 1.
    // It runs only where no attempt has left D(y) (the start of a solve, after a
    // change of the operator or a projection of rho_0); elsewhere the step pass forms
    // that input from the stored D.  Stage i (0-based, 1..5) evaluates k_{i+1} at its
    // input and writes the input of stage i+1 (rkdp.h:111-127); stage 5 forms the new
    // state (rkdp.h:130-132) and, from the same operands, the error sum
    // e6 = sum_{j<6} E_j k_j in the order of rkdp.h:142-145 (k_6 itself is
    // not stored); stage 6 evaluates D at the new state, stores it as the next
    // attempt's stage 0, completes e = e6 + E_7 k_7 and the error norm
    // (rkdp.h:144-153).  The error vector is the same fma chain as summing all
    // seven terms in the last stage.
    const int sin_[6] = {y_in, SL_SA, SL_SB, SL_SA, SL_SB, SL_SA};
    const int sout[5] = {SL_SA, SL_SB, SL_SA, SL_SB, SL_SA};
    const auto k_of = [](int j) { return j == 0 ? int(SL_D) : SL_K1 + j; };
    for (int i = 0; i < 6; ++i) {
      StageSpec a;
      a.in_slot = sin_[i];
      std::vector<std::pair<int, double>> terms{{SL_Y, 1.0}};
      if (i == 0) {
        a.k_slot = SL_D;
        a.combo(terms, kDpA[1][0], sout[0]);
      } else if (i < 5) {
        a.k_slot = SL_K1 + i;
        for (int j = 0; j < i; ++j) terms.push_back({k_of(j), kDpA[i + 1][j]});
        a.combo(terms, kDpA[i + 1][i], sout[i]);
      } else {
        for (int j = 0; j < 5; ++j)
          if (kDpB[j] != 0.0) terms.push_back({k_of(j), kDpB[j]});
        a.combo(terms, kDpB[5], SL_YNEW, lo ? SL_YNEW32 : -1);
        std::vector<std::pair<int, double>> eterms;
        for (int j = 0; j < 5; ++j)
          if (kDpE[j] != 0.0) eterms.push_back({k_of(j), kDpE[j]});
        a.combo(eterms, kDpE[5], SL_E);
      }
      specs.push_back(a);
    }
    StageSpec a;
    a.in_slot = lo ? SL_YNEW32 : SL_YNEW;
    a.k_slot = SL_DNEW;
    a.do_err = 1;
    a.ek = kDpE[6];
    a.pre = {SL_E, SL_YNEW, SL_Y};  // as the epilogue takes them
    specs.push_back(a);
  }
  for (auto& s : specs) {
    StageArgs r = resolve(s);
    r.atol = atol;
    r.rtol = rtol;
    stages.push_back(r);
  }
}

// Whether (and with which compiled-in stage program) the resident integrator
// runs this fixed-step problem.
void Solver::build_resident() {
  res = ResidentArgs{};
  if (!use_resident || kind == HEOM_RKDP || in_bytes != 8 || q->opt.renorm_rho0 ||
      !resident_ok(q->dev, q->dev.max_links))
    return;
  const ResidentProg& P = kind == HEOM_RK4 ? kResidentRk4 : kResidentLsrk4;
  if (resident_lds_bytes(q->dev, P.n_buf) > kResidentLds) return;
  res.scheme = kind == HEOM_RK4 ? 1 : 2;
}

// Where a resident launch leaves its results in host memory (see ResidentHost)
ResidentHost Solver::resident_host() {
  if (h_state == nullptr)
    HAMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&h_state), sizeof(z128) * kResidentMax,
                           hipHostMallocCoherent));
  __atomic_store_n(mail, 0ull, __ATOMIC_RELEASE);
  return ResidentHost{h_state, h_ctrl, mail};
}

// Small problems: an interval per resident launch.  The levels for which a
// wavefront holds the same ADOs as a workgroup of the stage kernels: the
// error norm is then the same sum, so the steps are decided alike (spin-boson
// depth 6, ten intervals: 4.6 ms with the stage kernels, 0.52 ms here).
bool Solver::dopri_interval_resident() const {
  return use_resident && in_bytes == 8 && !q->opt.renorm_rho0 && q->dev.kind == HEOM_HILB &&
         (q->N == 1 || q->N == 2 || q->N == 4) && resident_dopri_ok(q->dev, q->dev.max_links);
}

// One Dormand-Prince interval of a small problem in one resident launch, as
// run_attempts: the state stays in slot SL_Y, the control block's counters add
// up over the intervals.
int Solver::rkdp_interval_resident(double t0, double t1, double dt_first, double atol,
                                   double rtol) {
  ResidentDopriArgs a{};
  a.y = static_cast<z128*>(P[SL_Y].p);
  a.n_int = 1;
  a.t0 = t0;
  a.t1 = t1;
  a.tree = 1;
  a.dt_first = dt_first;
  a.atol = atol;
  a.rtol = rtol;
  a.inv_n = 1.0 / static_cast<double>(ms);
  a.ctrl = d_ctrl.as<Ctrl>();
  const Ctrl before = *h_ctrl;
  a.host = resident_host();
  launch_resident_dopri(q->dev, q->dev.max_links, a, q->stream);
  (void)wait_mail(0);
  host_state = h_state;
  h_ctrl->cur = 0;
  h_ctrl->attempts += before.attempts;
  h_ctrl->accepted += before.accepted;
  h_ctrl->rejected += before.rejected;
  return h_ctrl->gave_up;
}

// rho_0 projection after a step / attempt (heom_options.renorm_rho0)
void Solver::renorm(bool with_ctrl) {
  const bool lo = in_bytes == 4;
  launch_rho0_renorm(slot_ptr(SL_Y, 0), slot_ptr(SL_Y, with_ctrl ? 1 : 0),
                     lo ? slot_ptr(SL_Y32, 0) : nullptr,
                     lo ? slot_ptr(SL_Y32, with_ctrl ? 1 : 0) : nullptr,
                     with_ctrl ? ctrl_dev() + par : nullptr, q->N, d_tr0.as<double>(), stream());
}

void Solver::launch_stage(int s, double dt) {
  StageArgs a = stages[s];
  a.a_re = dt;
  if (a.ctrl) a.ctrl += par;
  const int grid = q->operate(in_bytes, a, stream());
  if (a.do_err) n_partials = grid;
}

// A run of many short stages waits longer between its kernels when the host launches
// them one by one (RK4, 16 000 stages of 364 ADOs of 2x2: 4.80 us per stage, 4.41 from
// graphs), but a graph costs its instantiation, some 100 us, on every solve: fixed steps
// are replayed in graphs of up to kGraphSteps steps when the solve makes kGraphReplays or
// more of them, Dormand-Prince attempts one at a time after kGraphAttempts of them.  70 ADOs
// of 5x5, RK4, intervals x steps, launched -> graphs of 8 (of 16): 1 x 32 0.76 -> 0.85 (0.95)
// ms, 1 x 128 2.98 -> 2.66 (2.71), 10 x 10 2.69 -> 2.43 (2.68), 10 x 40 9.66 -> 8.20 (8.18);
// graphs of 4, 10 x 5 1.53 -> 1.36; graphs of 2, 100 x 3 10.2 -> 8.3.  Longer stages
// hide the host's launches, and then a graph's start costs more than it saves: RK4 step and
// attempt of 253 ADOs of 7x7 18.7 -> 17.7 and 42.3 -> 39.0 us, 2024 ADOs (99 000 elements)
// 21.5 and 44.8 -> 21.4 and 45.3, 12 650 ADOs 60.9 and 122.4 -> 61.6 and 126.9; RK4 step of
// 80 000 elements in 4x4 31.2 -> 30.1, of 167 000 in 3x3 42.3 -> 42.9.  Fixed steps of
// more than kGraphAttemptSize elements therefore have to make eight times the replays.
constexpr int kGraphSteps = 8, kGraphReplays = 8, kGraphAttempts = 128;
constexpr long long kGraphStepSize = 1 << 17, kGraphAttemptSize = 1 << 16;  // elements

// Launch `body` from graph `key`, which is recorded the first time.  The body launches
// kernels only (no copy or memset: replays of memset nodes have gone wrong).
void Solver::replay(int key, const std::function<void()>& body) {
  GraphExec& g = graphs[key];
  if (g.exec == nullptr) {
    if (rec_stream == nullptr)
      HAMD_HIP(hipStreamCreateWithFlags(&rec_stream, hipStreamNonBlocking));
    HAMD_HIP(hipStreamBeginCapture(rec_stream, hipStreamCaptureModeThreadLocal));
    hipGraph_t graph = nullptr;
    recording = true;
    try {
      body();
    } catch (...) {
      recording = false;
      (void)hipStreamEndCapture(rec_stream, &graph);
      if (graph) (void)hipGraphDestroy(graph);
      throw;
    }
    recording = false;
    HAMD_HIP(hipStreamEndCapture(rec_stream, &graph));
    const hipError_t e = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    HAMD_HIP(e);
  }
  HAMD_HIP(hipGraphLaunch(g.exec, q->stream));
}

// fixed_step_size_solver::solve_1 (fixed_step_size_solver.h:29-52): steps of
// dt, the last one shortened to end exactly at t1.  The step sequence is
// computed on the host with the reference's arithmetic.
void Solver::fixed_steps(double t0, double t1, double dt, long long& n_full, double& dt_last) {
  double t = t0, dt_1 = dt;
  n_full = 0;
  while (true) {
    if (t + dt_1 - t1 > -std::numeric_limits<double>::epsilon()) {
      dt_1 = t1 - t;
      break;
    }
    ++n_full;
    t += dt_1;
  }
  dt_last = dt_1;
}

// Steps per graph of a solve, 0 for none: the largest power of two that an interval holds,
// when it is replayed kGraphReplays times `scale` or more
int Solver::graph_size(const double* t_list, int n_t, double dt, int scale) {
  std::vector<long long> n(n_t > 1 ? n_t - 1 : 0);
  double last = 0.0;
  for (int i = 0; i + 1 < n_t; ++i) fixed_steps(t_list[i], t_list[i + 1], dt, n[i], last);
  const long long longest = n.empty() ? 0 : *std::max_element(n.begin(), n.end());
  int size = kGraphSteps;
  while (size > 1 && size > longest) size /= 2;
  if (size < 2) return 0;
  long long replays = 0;
  for (const long long k : n) replays += k / size;
  return replays >= kGraphReplays * scale ? size : 0;
}

void Solver::rk4_interval(double t0, double t1, double dt) {
  long long n_full = 0;
  double dt_1 = dt;
  fixed_steps(t0, t1, dt, n_full, dt_1);
  if (res.scheme != 0) {  // the whole interval in one launch
    ResidentArgs a = res;
    a.y = static_cast<z128*>(P[SL_Y].p);
    a.n_full = n_full;
    a.dt = dt;
    a.dt_last = dt_1;
    if (to_host) a.host = resident_host();
    launch_resident(q->dev, q->dev.max_links, a, q->stream);
    if (to_host) {
      (void)wait_mail(0);
      host_state = h_state;
    }
    stats.n_rhs += 4 * (n_full + 1);
    stats.n_attempts += n_full + 1;
    stats.n_accepted += n_full + 1;
    return;
  }
  const auto step = [&] {
    for (int s = 0; s < 4; ++s) launch_stage(s, dt);
    if (q->opt.renorm_rho0) renorm(false);
  };
  for (long long n = 0; n < n_full;) {
    const int size = graph_steps > 0 && graph_warm && n_full - n >= graph_steps ? graph_steps : 1;
    if (size > 1)
      replay(size, [&] {
        for (int k = 0; k < size; ++k) step();
      });
    else
      step();
    graph_warm = true;
    n += size;
  }
  for (int s = 0; s < 4; ++s) launch_stage(s, dt_1);  // the last (shortened) step
  if (q->opt.renorm_rho0) renorm(false);
  stats.n_rhs += 4 * (n_full + 1);
  stats.n_attempts += n_full + 1;
  stats.n_accepted += n_full + 1;
}

// The pass between two attempts, see StepArgs
StepArgs Solver::step_args(int mode) const {
  StepArgs a{};
  a.mode = mode;
  a.next = ctrl_dev() + par;
  a.prev = (mode & STEP_CONTROL) ? ctrl_dev() + (par ^ 1) : a.next;
  a.partials = partials_dev();
  a.nparts = n_partials;
  a.inv_n = 1.0 / static_cast<double>(ms);
  a.t_list = step_t;
  a.n_int = step_n_int;
  a.rho_s = (mode & STEP_CONTROL) ? step_rho_s : nullptr;
  a.n_rs = q->N2;
  for (int cur = 0; cur < 2; ++cur) {
    a.y[cur] = static_cast<const z128*>(slot_ptr(SL_Y, cur));
    a.D[cur] = slot_ptr(SL_D, cur);
  }
  a.lo = in_bytes == 4 ? 1 : 0;
  a.sa = sp[SL_SA];
  a.a21 = kDpA[1][0];
  a.n = ms;
  a.mail = mail;
  return a;
}

void Solver::launch_step(int mode) {
  if (mode & STEP_CONTROL) par ^= 1;
  launch_dopri_step(step_args(mode), stream());
}

// The device's progress word once it has moved past `seen` step passes.
unsigned long long Solver::wait_mail(unsigned long long seen) {
  for (unsigned n = 1;; ++n) {
    const unsigned long long v = __atomic_load_n(mail, __ATOMIC_ACQUIRE);
    if ((v >> 2) > seen) return v;
    if (n % (1u << 14) == 0) std::this_thread::yield();
    if (n % (1u << 20) == 0) {
      const hipError_t e = hipStreamQuery(q->stream);
      if (e == hipErrorNotReady) continue;
      HAMD_HIP(e);
      // the stream has drained: the word is final
      const unsigned long long w = __atomic_load_n(mail, __ATOMIC_ACQUIRE);
      if ((w >> 2) > seen) return w;
      throw HeomError{HEOM_ERR_HIP, "rkdp: the step pass left no progress word"};
    }
  }
}

// Attempts of rkdp::solve_adaptive_step until the control block is done: one
// output interval (adaptive_step_size_solver::solve_1,
// adaptive_step_size_solver.h:32-56), or all of step_t.  While an attempt runs,
// the next one is queued behind it, so the device never waits for the host; when
// the running attempt can be the last, only its step pass is, so that nothing is
// left over (attempts queued in batches left 3-4 idle ones per solve of 30).
// stale: SL_D is not D of the state the first attempt starts from.
int Solver::run_attempts(bool stale) {
  const bool proj = q->opt.renorm_rho0 != 0;
  __atomic_store_n(mail, 0ull, __ATOMIC_RELEASE);
  // a projection of rho_0 (after every attempt; it acts only on an accepted one)
  // makes the stored D stale.  Stage 0 then takes the place of the step pass's stream:
  // 7-site chain, projected, 1 ps: 136.5 us per attempt (FP64 147.4) with stage 0 storing D
  // alone and a launch more for the stage input, 127.4 us (FP64 136.9)
  const auto step = [&](bool first) {
    const bool eval = proj || (first && stale);
    launch_step(STEP_CONTROL | (first ? STEP_FIRST : 0) | (eval ? 0 : STEP_INPUT));
    if (proj && !first) renorm(true);
    if (eval) launch_stage(0, 0.0);
  };
  const auto evaluate = [&] {
    for (int s = 1; s < 7; ++s) launch_stage(s, 0.0);
  };
  step(true);
  evaluate();
  unsigned long long steps = 1, attempts = 1, seen = 0;
  while (true) {
    const unsigned long long v = wait_mail(seen);
    seen = v >> 2;
    if (v & 1) break;
    if (attempts < seen) {  // the attempt held back as possibly not needed
      evaluate();
      ++attempts;
      ++direct_attempts;
    }
    if (use_resident && ms <= kGraphAttemptSize && direct_attempts >= kGraphAttempts &&
        !(v & 2) && steps < seen + 1 && attempts == steps) {
      const int from = par;  // the step pass writes the other control block
      replay(from, [&] {
        step(false);
        evaluate();
      });
      par = from ^ 1;
      ++steps;
      ++attempts;
    }
    if (steps < seen + 1) {
      step(false);
      ++steps;
    }
    if (!(v & 2) && attempts < seen + 1) {
      evaluate();
      ++attempts;
      ++direct_attempts;
    }
  }
  HAMD_HIP(hipMemcpyAsync(h_ctrl, ctrl_dev() + par, sizeof(Ctrl), hipMemcpyDeviceToHost,
                          q->stream));
  HAMD_HIP(hipStreamSynchronize(q->stream));
  return h_ctrl->gave_up;
}

void Solver::add_dopri_stats() {
  // the scheme's seven stages per attempt (the first one taken from the attempt
  // before it)
  stats.n_rhs += 7 * h_ctrl->attempts;
  stats.n_attempts += h_ctrl->attempts;
  stats.n_accepted += h_ctrl->accepted;
  stats.n_rejected += h_ctrl->rejected;
  stats.last_err = h_ctrl->err;
  stats.last_dt = dt_save;
}

int Solver::solve(void* rho_dev, const double* t_list, int n_t, double dt, double atol,
                  double rtol, const std::function<void(int, const void*)>& on_output) {
  check_qme();
  if (n_t < 1) throw HeomError{HEOM_ERR_ARG, "solve: n_t < 1"};
  for (int i = 0; i + 1 < n_t; ++i)
    if (!(t_list[i + 1] >= t_list[i]))
      throw HeomError{HEOM_ERR_ARG, "solve: t_list must be non-decreasing"};
  if (kind != HEOM_RKDP && !(dt > 0.0))
    throw HeomError{HEOM_ERR_ARG, "rk4/lsrk4: dt must be > 0"};
  if (kind == HEOM_RKDP) {
    if (!(dt > 0.0) && dt_save <= 0.0) throw HeomError{HEOM_ERR_ARG, "rkdp: dt must be > 0"};
    if (!(atol >= 0.0) || !(rtol >= 0.0) || (atol == 0.0 && rtol == 0.0))
      throw HeomError{HEOM_ERR_ARG, "rkdp: atol/rtol must be >= 0 and not both 0"};
  }
  HAMD_HIP(hipSetDevice(q->opt.device));
  build_stages(atol, rtol);
  build_resident();
  host_state = nullptr;
  const size_t bytes = sizeof(z128) * ms;
  hipStream_t st = q->stream;
  // the caller's state enters the FP64 state slot
  HAMD_HIP(hipMemcpyAsync(P[SL_Y].p, rho_dev, bytes, hipMemcpyDeviceToDevice, st));
  if (in_bytes == 4) launch_narrow(P[SL_Y32].p, P[SL_Y].p, ms, st);
  if (q->opt.renorm_rho0) launch_rho0_trace(P[SL_Y].p, q->N, d_tr0.as<double>(), st);
  int gave_up = 0;
  unsigned long long gen = q->generation;
  if (kind != HEOM_RKDP) {  // fixed step: rk4, lsrk4
    graph_steps = use_resident && res.scheme == 0 && ms <= kGraphStepSize
                      ? graph_size(t_list, n_t, dt, ms <= kGraphAttemptSize ? 1 : 8)
                      : 0;
    for (int i = 0; i < n_t - 1; ++i) {
      on_output(i, P[SL_Y].p);
      if (operator_changed(gen)) {
        build_resident();
        if (res.scheme == 0) host_state = nullptr;
      }
      rk4_interval(t_list[i], t_list[i + 1], dt);
    }
    on_output(n_t - 1, P[SL_Y].p);
    HAMD_HIP(hipMemcpyAsync(rho_dev, P[SL_Y].p, bytes, hipMemcpyDeviceToDevice, st));
  } else {
    bool resident = dopri_interval_resident();
    std::memset(h_ctrl, 0, sizeof(Ctrl));
    double first = dt_save > 0.0 ? dt_save : dt;
    Ctrl before{};  // counters of resident intervals that stage launches continue
    int cur = 0;
    bool started = false;
    bool on_device = false;  // the device's control block carries the step size and counters
    bool stale = true;       // SL_D is not D of the current state and operator
    for (int i = 0; i < n_t - 1; ++i) {
      on_output(i, P[cur].p);
      if (operator_changed(gen)) {
        stale = true;
        if (resident && !dopri_interval_resident()) {
          resident = false;
          host_state = nullptr;
          if (started) first = h_ctrl->dt;
          before = *h_ctrl;
        }
      }
      // a zero-length interval takes no attempt and keeps the step size (the
      // reference would clamp the step to 0 and never finish the next interval)
      if (!(t_list[i + 1] > t_list[i])) continue;
      if (resident) {
        gave_up |= rkdp_interval_resident(t_list[i], t_list[i + 1], started ? h_ctrl->dt : first,
                                          atol, rtol);
      } else {
        launch_ctrl_init(ctrl_dev() + par, t_list[i], t_list[i + 1], on_device ? -1.0 : first, i,
                         st);
        gave_up |= run_attempts(stale);
        on_device = true;
        stale = false;
      }
      started = true;
      cur = h_ctrl->cur;
    }
    if (on_device) {
      h_ctrl->attempts += before.attempts;
      h_ctrl->accepted += before.accepted;
      h_ctrl->rejected += before.rejected;
    }
    on_output(n_t - 1, P[cur].p);
    if (started) dt_save = h_ctrl->dt;
    add_dopri_stats();
    HAMD_HIP(hipMemcpyAsync(rho_dev, P[cur].p, bytes, hipMemcpyDeviceToDevice, st));
  }
  HAMD_HIP(hipStreamSynchronize(st));
  graphs.clear();
  stats.ado_stage_updates = stats.n_rhs * q->hs.n_hrchy;
  stats.gave_up |= gave_up;
  return gave_up ? HEOM_ERR_STEP_REJECTED : HEOM_OK;
}

int Solver::solve_gather(void* rho_dev, const double* t_list, int n_t, double dt, double atol,
                         double rtol, void* rho_s_dev) {
  check_qme();
  const size_t rs_bytes = sizeof(z128) * q->N2;
  hipStream_t st = q->stream;
  if (kind == HEOM_RKDP && n_t >= 2 && !q->opt.renorm_rho0 && q->kind != kBatch)
    return solve_dopri(rho_dev, t_list, n_t, dt, atol, rtol, rho_s_dev);
  if (kind == HEOM_RKDP || n_t < 2 || q->kind == kBatch) {
    return solve(rho_dev, t_list, n_t, dt, atol, rtol, [&](int i, const void* cur) {
      HAMD_HIP(hipMemcpyAsync(static_cast<char*>(rho_s_dev) + rs_bytes * i, cur, rs_bytes,
                              hipMemcpyDeviceToDevice, st));
    });
  }
  for (int i = 0; i + 1 < n_t; ++i)
    if (!(t_list[i + 1] >= t_list[i]))
      throw HeomError{HEOM_ERR_ARG, "solve: t_list must be non-decreasing"};
  if (!(dt > 0.0)) throw HeomError{HEOM_ERR_ARG, "rk4/lsrk4: dt must be > 0"};
  HAMD_HIP(hipSetDevice(q->opt.device));
  build_stages(atol, rtol);
  build_resident();
  if (res.scheme == 0) {
    return solve(rho_dev, t_list, n_t, dt, atol, rtol, [&](int i, const void* cur) {
      HAMD_HIP(hipMemcpyAsync(static_cast<char*>(rho_s_dev) + rs_bytes * i, cur, rs_bytes,
                              hipMemcpyDeviceToDevice, st));
    });
  }
  // the whole solve in one resident launch
  std::vector<long long> nf(n_t - 1);
  std::vector<double> dl(n_t - 1);
  long long steps = 0;
  for (int i = 0; i + 1 < n_t; ++i) {
    fixed_steps(t_list[i], t_list[i + 1], dt, nf[i], dl[i]);
    steps += nf[i] + 1;
  }
  upload_kept(d_res_nf, nf.data(), sizeof(long long) * nf.size());
  upload_kept(d_res_dl, dl.data(), sizeof(double) * dl.size());
  ResidentArgs a = res;
  a.y = static_cast<z128*>(P[SL_Y].p);
  a.dt = dt;
  a.n_int = n_t - 1;
  a.n_full_i = d_res_nf.as<long long>();
  a.dt_last_i = d_res_dl.as<double>();
  a.rho_s = static_cast<z128*>(rho_s_dev);
  const size_t bytes = sizeof(z128) * ms;
  HAMD_HIP(hipMemcpyAsync(P[SL_Y].p, rho_dev, bytes, hipMemcpyDeviceToDevice, st));
  launch_resident(q->dev, q->dev.max_links, a, st);
  HAMD_HIP(hipMemcpyAsync(rho_dev, P[SL_Y].p, bytes, hipMemcpyDeviceToDevice, st));
  HAMD_HIP(hipStreamSynchronize(st));
  stats.n_rhs += 4 * steps;
  stats.n_attempts += steps;
  stats.n_accepted += steps;
  stats.ado_stage_updates = stats.n_rhs * q->hs.n_hrchy;
  return HEOM_OK;
}

// adaptive_step_size_solver::solve (adaptive_step_size_solver.h:32-56) with the
// device walking through the output times: a small problem in one resident
// launch, others as a queue of attempts without a stop between the intervals.
int Solver::solve_dopri(void* rho_dev, const double* t_list, int n_t, double dt, double atol,
                        double rtol, void* rho_s_dev) {
  check_qme();
  int first = -1;  // first interval of positive length
  for (int i = 0; i + 1 < n_t; ++i) {
    if (!(t_list[i + 1] >= t_list[i]))
      throw HeomError{HEOM_ERR_ARG, "solve: t_list must be non-decreasing"};
    if (first < 0 && t_list[i + 1] > t_list[i]) first = i;
  }
  if (!(dt > 0.0) && dt_save <= 0.0) throw HeomError{HEOM_ERR_ARG, "rkdp: dt must be > 0"};
  if (!(atol >= 0.0) || !(rtol >= 0.0) || (atol == 0.0 && rtol == 0.0))
    throw HeomError{HEOM_ERR_ARG, "rkdp: atol/rtol must be >= 0 and not both 0"};
  HAMD_HIP(hipSetDevice(q->opt.device));
  build_stages(atol, rtol);
  hipStream_t st = q->stream;
  const bool resident =
      use_resident && in_bytes == 8 && resident_dopri_ok(q->dev, q->dev.max_links);
  upload_times(t_list, n_t);
  const double dt_first = dt_save > 0.0 ? dt_save : dt;
  const size_t bytes = sizeof(z128) * ms;
  HAMD_HIP(hipMemcpyAsync(P[SL_Y].p, rho_dev, bytes, hipMemcpyDeviceToDevice, st));
  std::memset(h_ctrl, 0, sizeof(Ctrl));
  if (resident) {
    ResidentDopriArgs a{};
    a.y = static_cast<z128*>(P[SL_Y].p);
    a.n_int = n_t - 1;
    a.t_list = d_res_t.as<double>();
    a.dt_first = dt_first;
    a.atol = atol;
    a.rtol = rtol;
    a.inv_n = 1.0 / static_cast<double>(ms);
    a.rho_s = static_cast<z128*>(rho_s_dev);
    a.ctrl = d_ctrl.as<Ctrl>();
    launch_resident_dopri(q->dev, q->dev.max_links, a, st);
    HAMD_HIP(hipMemcpyAsync(rho_dev, P[SL_Y].p, bytes, hipMemcpyDeviceToDevice, st));
    HAMD_HIP(hipMemcpyAsync(h_ctrl, d_ctrl.p, sizeof(Ctrl), hipMemcpyDeviceToHost, st));
  } else if (first < 0) {  // outputs only
    for (int i = 0; i < n_t; ++i)
      HAMD_HIP(hipMemcpyAsync(static_cast<z128*>(rho_s_dev) + static_cast<size_t>(i) * q->N2,
                              P[SL_Y].p, sizeof(z128) * q->N2, hipMemcpyDeviceToDevice, st));
  } else {
    if (in_bytes == 4) launch_narrow(P[SL_Y32].p, P[SL_Y].p, ms, st);
    launch_ctrl_init(ctrl_dev() + par, t_list[first], t_list[first + 1], dt_first, first, st);
    step_t = d_res_t.as<double>();
    step_n_int = n_t - 1;
    step_rho_s = static_cast<z128*>(rho_s_dev);
    try {
      run_attempts(true);
    } catch (...) {
      step_t = nullptr;
      step_rho_s = nullptr;
      throw;
    }
    step_t = nullptr;
    step_rho_s = nullptr;
    HAMD_HIP(hipMemcpyAsync(rho_dev, P[h_ctrl->cur].p, bytes, hipMemcpyDeviceToDevice, st));
  }
  HAMD_HIP(hipStreamSynchronize(st));
  graphs.clear();
  // only intervals of positive length touch the step size (as in solve)
  if (first >= 0) dt_save = h_ctrl->dt;
  add_dopri_stats();
  stats.ado_stage_updates = stats.n_rhs * q->hs.n_hrchy;
  stats.gave_up |= h_ctrl->gave_up;
  return h_ctrl->gave_up ? HEOM_ERR_STEP_REJECTED : HEOM_OK;
}

int Solver::solve_noalloc(void* rho_dev, const double* t_list, int n_t, double dt, double atol,
                          double rtol, Ctrl* ctrl, double* partials, void* rho_s_dev) {
  check_qme();
  if (q->closure) throw HeomError{HEOM_ERR_UNSUPPORTED, "solve_noalloc: a closure is bound"};
  const bool batch = q->kind == kBatch;
  const size_t rs_bytes = sizeof(z128) * (batch ? q->batch_rs_size : q->N2);
  hipStream_t st = q->stream;
  const bool resident = use_resident;
  use_resident = false;
  ext_ctrl = ctrl;
  ext_partials = partials;
  int rc = HEOM_OK;
  try {
    rc = solve(rho_dev, t_list, n_t, dt, atol, rtol, [&](int i, const void* cur) {
      char* dst = static_cast<char*>(rho_s_dev) + rs_bytes * i;
      if (batch)
        launch_gather_rho_s(q->dev, dst, cur, st);
      else
        HAMD_HIP(hipMemcpyAsync(dst, cur, rs_bytes, hipMemcpyDeviceToDevice, st));
    });
  } catch (...) {
    use_resident = resident;
    ext_ctrl = nullptr;
    ext_partials = nullptr;
    throw;
  }
  use_resident = resident;
  ext_ctrl = nullptr;
  ext_partials = nullptr;
  return rc;
}

void Solver::time_stages(int reps, std::vector<double>& out) {
  check_qme();
  HAMD_HIP(hipSetDevice(q->opt.device));
  hipStream_t st = q->stream;
  const int ns = n_stages();
  out.assign(ns, 0.0);
  if (kind == HEOM_RKDP) {
    // a control block that never finishes: every pass, the step pass too, starts from it
    Ctrl c{};
    c.t = 0.0;
    c.t_bound = 1e300;
    c.dt = dt_save > 0.0 ? dt_save : 1e-3;
    c.cur = h_ctrl ? h_ctrl->cur : 0;
    std::memcpy(h_ctrl, &c, sizeof(Ctrl));
    par = 0;
    HAMD_HIP(hipMemcpyAsync(d_ctrl.p, h_ctrl, sizeof(Ctrl), hipMemcpyHostToDevice, st));
    n_partials = launch_operator(q->dev, in_bytes, stages[6], st);  // what the step pass adds up
  }
  hipEvent_t e0, e1;
  HAMD_HIP(hipEventCreate(&e0));
  HAMD_HIP(hipEventCreate(&e1));
  for (int s = 0; s < ns; ++s) {
    StageArgs a = stages[s];
    a.a_re = 1e-3;
    // the first of the seven Dormand-Prince passes is the step pass with its decision
    // (with a projection of rho_0: stage 0); the decision goes to the other control block
    const auto pass = [&] {
      if (kind == HEOM_RKDP && s == 0 && !q->opt.renorm_rho0) {
        StepArgs sa = step_args(STEP_CONTROL | STEP_INPUT);
        sa.prev = ctrl_dev();
        sa.next = ctrl_dev() + 1;
        launch_dopri_step(sa, st);
      } else {
        launch_operator(q->dev, in_bytes, a, st);
      }
    };
    pass();  // warm-up
    HAMD_HIP(hipEventRecord(e0, st));
    for (int r = 0; r < reps; ++r) pass();
    HAMD_HIP(hipEventRecord(e1, st));
    HAMD_HIP(hipEventSynchronize(e1));
    float msf = 0.f;
    HAMD_HIP(hipEventElapsedTime(&msf, e0, e1));
    out[s] = static_cast<double>(msf) / reps;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
}

// Algorithmic HBM bytes of each stage pass: every state-sized buffer the
// pass reads or writes counts once per element (neighbour reads of the stage
// input are another ADO's compulsory read), plus the operator tables.
void Solver::stage_bytes(std::vector<double>& out) {
  const int ns = n_stages();
  out.assign(ns, 0.0);
  auto size_of = [&](int slot) { return slo[slot] ? 8.0 : 16.0; };
  double tables = 0.0;
  if (q->kind == HEOM_REDFIELD_LIOU) {
    tables = 20.0 * q->csr_nnz + 8.0 * (ms + 1);
  } else if (q->kind == HEOM_REDFIELD_HILB) {
    // H, and V_u, Lambda_u, Lambda_u^+ per noise
    tables = 16.0 * q->N2 * (1.0 + 3.0 * static_cast<double>(q->noise.size()));
  } else {
    // the fast Hilbert kernel (diagonal V, 6 <= N <= 16) reads 8-byte links and
    // the coefficient table, the other diagonal-V Hilbert kernels LinkFlat
    const bool fast = q->dev.kind == HEOM_HILB && q->dev.diag_v && q->N >= 6 && q->N <= 16;
    const double lrec = q->kind == kBatch || fast           ? sizeof(Link)
                        : (q->dev.kind == HEOM_HILB && q->dev.diag_v) ? sizeof(LinkFlat)
                                                               : sizeof(Link);
    tables = lrec * q->n_links + 4.0 * (q->hs.n_hrchy + 1) + 16.0 * q->hs.n_hrchy;
    if (q->kind == kBatch)
      tables += (q->lo() ? sizeof(BatchCoef<float>) : sizeof(BatchCoef<double>)) *
                    static_cast<double>(q->batch_n_coef) +
                sizeof(BatchItem) * static_cast<double>(q->dev.n_items);
    if (fast) tables += sizeof(Coef) * static_cast<double>(q->coef.size());
  }
  for (int s = 0; s < ns; ++s) {
    const StageSpec& a = specs[s];
    std::set<int> rd, wr;
    rd.insert(a.in_slot);
    for (int j : a.pre)
      if (j >= 0) rd.insert(j);
    if (a.k_slot >= 0) wr.insert(a.k_slot);
    for (int c = 0; c < a.ncombo; ++c) {
      wr.insert(a.dst[c]);
      if (a.dst2[c] >= 0) wr.insert(a.dst2[c]);
    }
    double per = 0.0;
    for (int r : rd) per += size_of(r);
    for (int w : wr) per += size_of(w);
    out[s] = per * static_cast<double>(ms) + tables;
    // the step pass: y and D read, the next stage input written
    if (kind == HEOM_RKDP && s == 0 && !q->opt.renorm_rho0)
      out[s] = (16.0 + size_of(SL_D) + size_of(SL_SA)) * static_cast<double>(ms);
  }
}

}  // namespace hamd
