// Runge-Kutta drivers with device-resident state (solver/*.h of the reference).
#pragma once

#include <functional>
#include <map>
#include <memory>
#include <vector>

#include "qme.h"

namespace hamd {

// Slot-level description of one stage pass; resolved into a StageArgs with
// device pointers for both ping-pong parities.
struct StageSpec {
  int in_slot = 0;
  int k_slot = -1;
  std::vector<int> pre;  // operand slots, in summation order
  int ncombo = 0;
  double cc[2][kMaxPre] = {};
  double ck[2] = {};
  int dst[2] = {-1, -1};
  int dst2[2] = {-1, -1};
  int do_err = 0;
  double ek = 0.0;
  int pre_index(int slot);
  void combo(const std::vector<std::pair<int, double>>& terms, double ckv, int d, int d2 = -1);
};

// An instantiated graph, destroyed with the object.
struct GraphExec {
  hipGraphExec_t exec = nullptr;
  GraphExec() = default;
  GraphExec(const GraphExec&) = delete;
  GraphExec& operator=(const GraphExec&) = delete;
  ~GraphExec() {
    if (exec) (void)hipGraphExecDestroy(exec);
  }
};

class Solver {
 public:
  Solver(std::shared_ptr<Qme> q, int kind);
  ~Solver();

  std::shared_ptr<Qme> q_owner;  // keeps the QME alive while the solver exists
  Qme* q;
  int kind;        // HEOM_RK4 / HEOM_RKDP / HEOM_LSRK4
  int in_bytes;    // real size of the operator arithmetic and stage inputs (8 or 4)
  long long ms;    // main_size
  double dt_save = -1.0;
  heom_stats stats{};
  // small problems in the resident integrators and long runs from graphs; false
  // launches every stage kernel
  bool use_resident = true;

  // Propagate the FP64 device state rho_dev over t_list.  on_output(i, cur_ptr)
  // is called at every t_i with a device pointer to the FP64 state.
  int solve(void* rho_dev, const double* t_list, int n_t, double dt, double atol, double rtol,
            const std::function<void(int, const void*)>& on_output);
  // The same with rho_S of every output time gathered into rho_s_dev (n_t N^2
  // complex128 in device memory) instead of a callback; a small problem then
  // runs the whole solve in one resident launch, and Dormand-Prince passes from
  // interval to interval on the device.
  int solve_gather(void* rho_dev, const double* t_list, int n_t, double dt, double atol,
                   double rtol, void* rho_s_dev);

  // solve_gather without any device allocation, for callers that cannot
  // allocate: every stage kernel is launched (no resident
  // integrator), the control blocks (two) and the error-norm partials are the
  // caller's (ctrl, partials: kMaxGrid doubles), and rho_S of every output time
  // is copied to rho_s_dev.  No closure may be bound.
  int solve_noalloc(void* rho_dev, const double* t_list, int n_t, double dt, double atol,
                    double rtol, Ctrl* ctrl, double* partials, void* rho_s_dev);

  // heom_solve: the resident launches leave the state in host memory as well.
  // host_state: the current state there, null when the output has to copy it
  bool to_host = false;
  const z128* host_state = nullptr;

  // device workspace of one solve call: the solver's d_state / d_rho_s while it is
  // at most kKeepWork bytes, else the caller's `own`
  static constexpr size_t kKeepWork = size_t(64) << 20;
  DevBuf d_state, d_rho_s;
  void* workspace(DevBuf& kept, DevBuf& own, size_t bytes);

  // Average duration (ms) of each stage kernel over `reps` replays.
  void time_stages(int reps, std::vector<double>& ms_out);
  // throws HEOM_ERR_STATE unless the QME is set up with the size the solver's
  // buffers were allocated for (set_param may have been called again)
  void check_qme() const;
  // whether a callback has changed the operator since `gen` (then moved on); the new
  // one must fit this solver's buffers
  bool operator_changed(unsigned long long& gen);
  void stage_bytes(std::vector<double>& bytes_out);
  int n_stages() const { return kind == HEOM_RKDP ? 7 : 4; }

 private:
  static constexpr int kSlots = 16;
  // slot table: slots 0..3 are ping-pong pairs (see common.h), resolved per
  // parity when a stage's pointers are built
  DevBuf P[kSlots];
  void* sp[kSlots] = {};
  int slo[kSlots] = {};  // 1: complex64 buffer
  DevBuf d_ctrl, d_partials;
  // control blocks and partials of the current solve (the solver's own, or a
  // caller's in solve_noalloc); the step passes read one block and write the
  // other, par is the one written last
  Ctrl* ext_ctrl = nullptr;
  double* ext_partials = nullptr;
  int par = 0;
  int n_partials = 0;  // partials of the last error-norm pass
  unsigned long long* mail = nullptr;  // progress word in pinned memory (see StepArgs)
  // output times the device walks through and where rho_S goes (null: one
  // interval at a time)
  const double* step_t = nullptr;
  int step_n_int = 0;
  z128* step_rho_s = nullptr;
  StepArgs step_args(int mode) const;
  void launch_step(int mode);
  unsigned long long wait_mail(unsigned long long seen);
  int run_attempts(bool stale);
  void add_dopri_stats();
  Ctrl* ctrl_dev() const { return ext_ctrl ? ext_ctrl : d_ctrl.as<Ctrl>(); }
  double* partials_dev() const { return ext_partials ? ext_partials : d_partials.as<double>(); }
  DevBuf d_tr0;  // Tr rho_0 at the start of the solve (renorm_rho0)
  void renorm(bool with_ctrl);
  Ctrl* h_ctrl = nullptr;  // pinned mirror
  std::vector<StageArgs> stages;

  void build_stages(double atol, double rtol);
  void* slot_ptr(int s, int cur) const;
  StageArgs resolve(const StageSpec& s) const;
  std::vector<StageSpec> specs;
  void launch_stage(int s, double dt);
  // Graphs of a long run's repeated launches (cleared when a solve begins and ends and
  // when the operator changes).  stream(): where launches go, the QME's stream or the one
  // that records a graph: a stream of its own that other threads' work on the default
  // stream does not wait for
  std::map<int, GraphExec> graphs;
  hipStream_t rec_stream = nullptr;
  bool recording = false;
  hipStream_t stream() const { return recording ? rec_stream : q->stream; }
  void replay(int key, const std::function<void()>& body);
  int graph_steps = 0;       // fixed steps of a graph of this solve, 0: none
  static int graph_size(const double* t_list, int n_t, double dt, int scale);
  bool graph_warm = false;   // a step of this operator has been launched (its kernels are loaded)
  long long direct_attempts = 0;  // Dormand-Prince: attempts of this solve launched one by one
  void rk4_interval(double t0, double t1, double dt);
  // resident integrator (small problems): scheme != 0 when the problem qualifies
  ResidentArgs res{};
  DevBuf d_res_nf, d_res_dl, d_res_t;
  double* h_times = nullptr;
  int n_times = 0;
  void upload_times(const double* t, int n);
  void upload_kept(DevBuf& b, const void* src, size_t bytes);
  z128* h_state = nullptr;  // pinned copy of a resident launch's state
  ResidentHost resident_host();
  int rkdp_interval_resident(double t0, double t1, double dt_first, double atol, double rtol);
  int solve_dopri(void* rho_dev, const double* t_list, int n_t, double dt, double atol,
                  double rtol, void* rho_s_dev);
  // fixed_step_size_solver::solve_1's step sequence over [t0, t1]: n_full steps
  // of dt, then one step of dt_last
  static void fixed_steps(double t0, double t1, double dt, long long& n_full, double& dt_last);
  void build_resident();
  // whether heom_solve runs Dormand-Prince intervals of this problem in resident launches
  bool dopri_interval_resident() const;
};

}  // namespace hamd
