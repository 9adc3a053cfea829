// Host runtime and C ABI of the MI355X FastMonodomainSolver fibre library.
//
// One shared library per cell model: the model header is selected at compile
// time (FMS_MODEL_HEADER / FMS_MODEL_TYPE), the way the reference compiles one
// library per CellML file (fast_monodomain_solver_gpu.tpp:12-206) - here ahead
// of time with hipcc for gfx950 instead of g++ -fopenmp at run time.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <type_traits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <new>
#include <string>
#include <vector>

#include "../../include/opendihu_fms.h"
#include "fms_fused.h"
#include "fms_kernels.h"
#include "fms_parts.h"


namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string &msg) {
  try {
    g_last_error = msg;
  } catch (...) {
    // no memory for the message: the code still reports the failure
  }
  return code;
}

// Every extern "C" entry runs its body inside FMS_API_BEGIN / FMS_API_END: a
// C++ exception (a host allocation that fails, ...) becomes FMS_ERR_INTERNAL
// and a message in fms_last_error instead of unwinding across the C ABI.
int api_exception() noexcept {
  try {
    throw;
  } catch (const std::bad_alloc &) {
    return fail(FMS_ERR_INTERNAL, "host memory allocation failed");
  } catch (const std::exception &e) {
    return fail(FMS_ERR_INTERNAL, std::string("internal error: ") + e.what());
  } catch (...) {
    return fail(FMS_ERR_INTERNAL, "internal error: unknown C++ exception");
  }
}

#define FMS_API_BEGIN try {
#define FMS_API_END                                                                                \
  }                                                                                                \
  catch (...) {                                                                                    \
    return api_exception();                                                                        \
  }
#define FMS_API_END_VOID                                                                           \
  }                                                                                                \
  catch (...) {                                                                                    \
    (void)api_exception();                                                                         \
  }

#define HIP_TRY(expr)                                                                              \
  do {                                                                                             \
    hipError_t e_ = (expr);                                                                        \
    if (e_ != hipSuccess)                                                                          \
      return fail(FMS_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));                 \
  } while (0)

template <class T> int dalloc(T **p, size_t n) {
  *p = nullptr;
  if (n == 0) n = 1;
  HIP_TRY(hipMalloc((void **)p, n * sizeof(T)));
  return 0;
}

template <class T> int h2d(T *d, const T *h, size_t n, hipStream_t s) {
  if (n == 0) return 0;
  HIP_TRY(hipMemcpyAsync(d, h, n * sizeof(T), hipMemcpyHostToDevice, s));
  return 0;
}

constexpr int FUSED_T = 256;
constexpr int PART_T = 256;

}  // namespace

struct FmsSolver {
  // configuration
  int F = 0;
  long long N = 0;
  long long GS = 0;   // gate stride: N rounded up to 64 nodes (every gate array 512-byte aligned)
  int scheme = FMS_IMPLICIT_EULER, precision = FMS_FP64, exp_mode = FMS_EXP_APPROXIMATE;
  int thomas = FMS_THOMAS_PARTITIONED, kernels = FMS_KERNELS_SPLIT;
  double vstim = 20.0;
  int nmax = 0;
  std::vector<int> h_off;     // [F+1]
  std::vector<int> h_order;   // fibres longest first
  int device = 0;             // the device current at fms_create
  hipStream_t stream = nullptr;
  hipStream_t stream2 = nullptr;   // adjoint: recompute of the next segment beside the reverse of this one
  hipEvent_t adj_ev[4] = {};

  // device state
  int *d_off = nullptr, *d_node_fiber = nullptr, *d_sb = nullptr, *d_se = nullptr, *d_order = nullptr;
  double *d_h = nullptr, *d_pf = nullptr, *d_params = nullptr;
  double *d_vm = nullptr;
  void *d_gates = nullptr;    // double or float [(NS-1)*GS]
  double *d_cA = nullptr, *d_dA = nullptr;  // serial Thomas scratch (split kernels)
  unsigned char *d_flags = nullptr;
  bool noalloc = false;   // the running call may not allocate (fms_advance_schedule_noalloc)
  size_t flags_cap = 0;   // bytes
  double *d_steps = nullptr;
  int steps_cap = 0;

  // stimulation
  int stim_mode = FMS_STIM_NONE;
  unsigned char *d_fe = nullptr;
  int *d_mu = nullptr, *d_joff = nullptr, *d_jcnt = nullptr, *d_jidx = nullptr;
  double *d_freq = nullptr, *d_rep = nullptr, *d_beg = nullptr, *d_jit = nullptr, *d_last = nullptr,
         *d_curjit = nullptr;
  unsigned char *d_curr = nullptr, *d_hasbeen = nullptr;
  int *d_log_count = nullptr, *d_log_fiber = nullptr;
  double *d_log_time = nullptr;
  int log_cap = 0;
  double *d_onset = nullptr, *d_dur = nullptr, *d_amp = nullptr;
  int stim_param = 0;
  int only_if_stimulated = 0;
  int fe_rows = 1, fe_cols = 1;
  // the reference's point-buffer order (fms_set_point_buffer_order)
  int vc_width = 0;
  double vc_factor = 0.0;
  int *d_vc_centre = nullptr;

  // spikes
  int spikes = 0;
  double spike_th = 0.0;
  double *d_vprev = nullptr;
  int *d_sfirst = nullptr, *d_scount = nullptr;
  long long step_counter = 0;

  // schedule knobs (fms_set_tuning): steps per fused launch, gate residency,
  // threads per fibre workgroup, split steps per captured graph (0: no graph)
  int tune_chunk = 512;
  int tune_resident = -1;   // k_fused: -1 auto, 0 stream gates from HBM, 1 keep gates in registers
  int tune_threads = 256;
  int tune_graph = 0;
  int tune_reaction_fibre = 1;   // split kernels, large models: one workgroup per fibre for the reaction
  int tune_pair = 1;   // split kernels: the two reaction halves between two solves in one launch
  int tune_reaction_threads = 256;   // split kernels, per-fibre reaction: threads per fibre workgroup (64 or 256)
  int tune_adjoint = FMS_ADJOINT_SERIAL;    // adjoint backward: recompute beside the reverse sweep or before it
  int tune_adjoint_threads = 512;           // reverse sweep: 256 threads per fibre (up to 1024 nodes), else 512
  int tune_adjoint_tape = FMS_ADJOINT_TAPE_AUTO;   // the forward records the whole tape, or checkpoints

  // per-kernel timing (fms_set_tuning(FMS_TUNE_PROFILE_KERNELS)): a start and
  // a stop event bound to each launch (hipExtLaunchKernel: the events take the
  // kernel's own begin and end, not the stream's state around it), from a pool
  // of PROF_POOL pairs that is read back when it is full and by fms_kernel_times
  static constexpr int PROF_POOL = 256;
  int prof = 0;
  hipEvent_t prof_ev[2 * PROF_POOL] = {};
  int prof_kind[PROF_POOL] = {};
  int prof_pending = 0;   // pairs recorded and not read back
  int prof_slot = -1;     // pair of the launch being enqueued, or -1
  int prof_launched = 0;  // FMS_LAUNCH bound that pair to a kernel
  double prof_ms[FMS_KERNEL_CLASSES] = {};
  long long prof_n[FMS_KERNEL_CLASSES] = {};

  // step cursor of the split kernels and the captured graph of tune_graph split steps
  long long *d_cursor = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  std::vector<unsigned char> graph_sig;
  long long n_graph_captures = 0, n_graph_launches = 0;

  // timing: events on the solver's stream and launch counters
  hipEvent_t events[8] = {};
  long long n_launch_fused = 0, n_launch_reaction = 0, n_launch_thomas = 0;

  // sensors, traces and the adjoint (checkpoints every ckpt_interval steps and a
  // tape of two segments, or the whole forward's tape)
  int n_sensors = 0;
  int *d_sensor_nodes = nullptr;   // [F][S] fibre-local
  int *d_sensor_slot = nullptr;    // [N]
  double *d_trace = nullptr, *d_dtrace = nullptr;
  long long trace_cap = 0;
  double *d_ckpt = nullptr, *d_tape = nullptr, *d_lam = nullptr, *d_gacc = nullptr, *d_pfbar = nullptr,
         *d_grad = nullptr;
  long long ckpt_cap = 0, tape_cap = 0;
  std::vector<double> adj_steps;   // host copy of the last adjoint forward's step table
  int adj_n0D = 1, adj_interval = 0, adj_K = 0;
  int adj_whole = 0;   // the last adjoint forward recorded the whole tape

  // algebraics for transfer
  int *d_alg_idx = nullptr;
  int n_alg_idx = 0;
  double *d_alg = nullptr;

  fms::DevFibers fibers() const {
    fms::DevFibers f;
    memset(&f, 0, sizeof(f));
    f.n_fibers = F;
    f.n_total = N;
    f.gate_stride = GS;
    f.fiber_off = d_off;
    f.node_fiber = d_node_fiber;
    f.elem_len = d_h;
    f.prefactor = d_pf;
    f.params = d_params;
    f.stim_begin = d_sb;
    f.stim_end = d_se;
    return f;
  }

  fms::DevStim stim() const {
    fms::DevStim s;
    memset(&s, 0, sizeof(s));
    s.mode = stim_mode;
    s.fe_rows = fe_rows;
    s.fe_cols = fe_cols;
    s.firing_events = d_fe;
    s.motor_unit = d_mu;
    s.freq = d_freq;
    s.repeat = d_rep;
    s.enable_begin = d_beg;
    s.jitter = d_jit;
    s.jitter_off = d_joff;
    s.jitter_cnt = d_jcnt;
    s.last_check = d_last;
    s.cur_jitter = d_curjit;
    s.jitter_idx = d_jidx;
    s.currently = d_curr;
    s.has_been = d_hasbeen;
    s.log_count = log_cap > 0 ? d_log_count : nullptr;
    s.log_time = d_log_time;
    s.log_fiber = d_log_fiber;
    s.log_cap = log_cap;
    s.onset = d_onset;
    s.duration = d_dur;
    s.amplitude = d_amp;
    s.stim_param = stim_param;
    s.only_if_stimulated = only_if_stimulated;
    s.vc_width = vc_width;
    s.vc_factor = vc_factor;
    s.vc_centre = d_vc_centre;
    return s;
  }
};

namespace {

void free_all(FmsSolver *s) {
  void *ptrs[] = {s->d_off, s->d_node_fiber, s->d_sb, s->d_se, s->d_order, s->d_h, s->d_pf, s->d_params,
                  s->d_vm, s->d_gates, s->d_cA, s->d_dA, s->d_flags, s->d_steps, s->d_fe, s->d_mu,
                  s->d_joff, s->d_jcnt, s->d_jidx, s->d_freq, s->d_rep, s->d_beg, s->d_jit, s->d_last,
                  s->d_curjit, s->d_curr, s->d_hasbeen, s->d_log_count, s->d_log_fiber, s->d_log_time,
                  s->d_onset, s->d_dur, s->d_amp, s->d_vprev, s->d_sfirst, s->d_scount, s->d_alg_idx,
                  s->d_alg, s->d_sensor_nodes, s->d_sensor_slot, s->d_trace, s->d_dtrace, s->d_ckpt, s->d_tape,
                  s->d_lam, s->d_gacc, s->d_pfbar, s->d_grad, s->d_cursor, s->d_vc_centre};
  if (s->graph_exec) (void)hipGraphExecDestroy(s->graph_exec);
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  for (hipEvent_t e : s->events)
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : s->adj_ev)
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : s->prof_ev)
    if (e) (void)hipEventDestroy(e);
  if (s->stream2) (void)hipStreamDestroy(s->stream2);
  if (s->stream) (void)hipStreamDestroy(s->stream);
}

// ---------------------------------------------------------------------------
// launchers, templated over gate type and exp policy
// ---------------------------------------------------------------------------

fms::StepRef step_ref(const FmsSolver *s, int q) { return fms::StepRef{s->d_cursor, q}; }

fms::DevSpikes dev_spikes(const FmsSolver *s) {
  fms::DevSpikes spk;
  memset(&spk, 0, sizeof(spk));
  spk.enabled = s->spikes;
  spk.threshold = s->spike_th;
  spk.vm_prev = s->d_vprev;
  spk.first_step = s->d_sfirst;
  spk.count = s->d_scount;
  spk.step0 = (int)s->step_counter;
  return spk;
}

int ensure_flag_bytes(FmsSolver *s, size_t bytes) {
  if (s->flags_cap < bytes) {
    if (s->d_flags) HIP_TRY(hipFree(s->d_flags));
    s->d_flags = nullptr;
    s->flags_cap = 0;
    if (dalloc(&s->d_flags, bytes)) return FMS_ERR_HIP;
    s->flags_cap = bytes;
  }
  return 0;
}

// the flags of one reaction half, or of a pair of halves (second buffer half)
int ensure_flags(FmsSolver *s, int n0D) { return ensure_flag_bytes(s, (size_t)2 * s->F * n0D); }

// adds the durations of the recorded launches to their classes
void prof_drain(FmsSolver *s) {
  for (int i = 0; i < s->prof_pending; i++) {
    float ms = 0;
    if (hipEventSynchronize(s->prof_ev[2 * i + 1]) == hipSuccess &&
        hipEventElapsedTime(&ms, s->prof_ev[2 * i], s->prof_ev[2 * i + 1]) == hipSuccess) {
      s->prof_ms[s->prof_kind[i]] += ms;
      s->prof_n[s->prof_kind[i]]++;
    }
  }
  s->prof_pending = 0;
}

// duration of the one launch in its scope (enqueued with FMS_LAUNCH) when
// per-kernel timing is on; the host does not wait for it
struct KernelTimer {
  FmsSolver *s;
  int kind;
  KernelTimer(FmsSolver *s_, int kind_) : s(s_), kind(kind_) {
    if (!s->prof) return;
    if (s->prof_pending == FmsSolver::PROF_POOL) prof_drain(s);
    s->prof_slot = s->prof_pending;
    s->prof_launched = 0;
  }
  ~KernelTimer() {
    if (s->prof_slot < 0) return;
    if (s->prof_launched) {
      s->prof_kind[s->prof_slot] = kind;
      s->prof_pending++;
    }
    s->prof_slot = -1;
  }
};

// a kernel launch on the solver's stream, with the timing pair of its
// KernelTimer bound to it when per-kernel timing is on
#define FMS_LAUNCH(s, kernel, grid, block, lds, ...)                                                         \
  do {                                                                                                       \
    if ((s)->prof_slot >= 0) {                                                                               \
      hipExtLaunchKernelGGL(kernel, grid, block, lds, (s)->stream, (s)->prof_ev[2 * (s)->prof_slot],         \
                            (s)->prof_ev[2 * (s)->prof_slot + 1], 0, __VA_ARGS__);                           \
      (s)->prof_launched = 1;                                                                                \
    } else                                                                                                   \
      hipLaunchKernelGGL(kernel, grid, block, lds, (s)->stream, __VA_ARGS__);                                \
  } while (0)

// device step table: the K records of this call plus a copy of the last one
// (the fused kernel reads one record ahead); the cursor starts at row 0 with
// the current spike-step counter (the split kernels read it; the others do not)
int upload_steps(FmsSolver *s, const double *steps, int K, bool cursor = true) {
  if (s->steps_cap < 4 * (K + 1)) {
    if (s->d_steps) HIP_TRY(hipFree(s->d_steps));
    s->d_steps = nullptr;
    s->steps_cap = 4 * (K + 1);
    if (dalloc(&s->d_steps, (size_t)s->steps_cap)) return FMS_ERR_HIP;
  }
  HIP_TRY(hipMemcpyAsync(s->d_steps, steps, 4 * (size_t)K * sizeof(double), hipMemcpyHostToDevice, s->stream));
  HIP_TRY(hipMemcpyAsync(s->d_steps + 4 * (size_t)K, steps + 4 * (size_t)(K - 1), 4 * sizeof(double),
                         hipMemcpyHostToDevice, s->stream));
  if (!cursor) return 0;
  hipLaunchKernelGGL(fms::k_cursor_set, dim3(1), dim3(64), 0, s->stream, s->d_cursor, 0LL, s->step_counter,
                     (const double *)s->d_steps);
  HIP_TRY(hipGetLastError());
  return 0;
}

// the per-fibre reaction of a large model with the workgroup size of the schedule
template <class G, class E, bool PAIR>
void launch_reaction_fibre(FmsSolver *s, int q, int half, int n0D, const fms::DevSpikes &spk) {
  if (s->tune_reaction_threads == 64)
    FMS_LAUNCH(s, (fms::k_reaction_fibre<Model, G, E, 64, PAIR>), dim3(s->F), dim3(64), 0,
               s->fibers(), s->stim(), s->d_vm, (G *)s->d_gates, s->d_flags, step_ref(s, q), half, n0D,
               s->vstim, s->d_order, spk);
  else
    FMS_LAUNCH(s, (fms::k_reaction_fibre<Model, G, E, 256, PAIR>), dim3(s->F), dim3(256), 0,
               s->fibers(), s->stim(), s->d_vm, (G *)s->d_gates, s->d_flags, step_ref(s, q), half, n0D,
               s->vstim, s->d_order, spk);
}

template <class G, class E>
int launch_reaction(FmsSolver *s, int q, int half, int n0D, bool store_alg) {
  KernelTimer timer(s, FMS_KERNEL_REACTION);
  const int threads = 256;
  const long long blocks = (s->N + threads - 1) / threads;
  const fms::DevSpikes off{};
  if (Model::NS > 8 && !store_alg && s->tune_reaction_fibre && !s->vc_width) {
    launch_reaction_fibre<G, E, false>(s, q, half, n0D, off);
  } else if (store_alg)
    FMS_LAUNCH(s, (fms::k_reaction<Model, G, E, true>), dim3((unsigned)blocks), dim3(threads), 0,
               s->fibers(), s->stim(), s->d_vm, (G *)s->d_gates, s->d_flags, step_ref(s, q), half, n0D,
               s->vstim, s->d_alg, s->d_alg_idx, s->n_alg_idx, off);
  else
    FMS_LAUNCH(s, (fms::k_reaction<Model, G, E, false>), dim3((unsigned)blocks), dim3(threads), 0,
               s->fibers(), s->stim(), s->d_vm, (G *)s->d_gates, s->d_flags, step_ref(s, q), half, n0D,
               s->vstim, nullptr, s->d_alg_idx, s->n_alg_idx, off);
  HIP_TRY(hipGetLastError());
  s->n_launch_reaction++;
  return 0;
}

// the second reaction half of step q and the first of step q+1 in one launch,
// with the spike detector of step q between them
template <class G, class E>
int launch_reaction_pair(FmsSolver *s, int q, int n0D) {
  KernelTimer timer(s, FMS_KERNEL_REACTION_PAIR);
  const fms::DevSpikes spk = dev_spikes(s);
  if (Model::NS > 8 && s->tune_reaction_fibre && !s->vc_width) {
    launch_reaction_fibre<G, E, true>(s, q, 1, n0D, spk);
  } else {
    const int threads = 256;
    const long long blocks = (s->N + threads - 1) / threads;
    FMS_LAUNCH(s, (fms::k_reaction<Model, G, E, false, true>), dim3((unsigned)blocks), dim3(threads), 0,
               s->fibers(), s->stim(), s->d_vm, (G *)s->d_gates, s->d_flags, step_ref(s, q), 1, n0D, s->vstim,
               nullptr, s->d_alg_idx, s->n_alg_idx, spk);
  }
  HIP_TRY(hipGetLastError());
  s->n_launch_reaction++;
  return 0;
}

int launch_flags(FmsSolver *s, int q, int half, int n0D) {
  KernelTimer timer(s, FMS_KERNEL_OTHER);
  const int threads = 64;
  FMS_LAUNCH(s, fms::k_stim_flags, dim3((s->F + threads - 1) / threads), dim3(threads), 0,
             s->stim(), s->F, s->d_flags, step_ref(s, q), half, n0D);
  HIP_TRY(hipGetLastError());
  return 0;
}

int launch_flags_pair(FmsSolver *s, int q, int n0D) {
  KernelTimer timer(s, FMS_KERNEL_OTHER);
  const int threads = 64;
  FMS_LAUNCH(s, fms::k_stim_flags_pair, dim3((s->F + threads - 1) / threads), dim3(threads), 0,
             s->stim(), s->F, s->d_flags, step_ref(s, q), n0D);
  HIP_TRY(hipGetLastError());
  return 0;
}

// Threads per fibre of the chunked kernels. Every kernel of the solver takes the
// same, so that its schedules agree in every bit. A thread owns ceil(n / T) <= 8
// nodes; 512 only for the fibres that need them: with 256, two fibres share a CU and
// one's solve hides behind the other's reaction (4096 fibres of 400-2000 nodes: 80
// against 109 us per step), and with one fibre per CU they differ by a few per cent
// in either direction (256 x 1000 nodes: both 6.1 us; 16 x 600: 4.6 against 5.3).
int chunk_threads(const FmsSolver *s) {
  if (s->tune_threads == 128 && s->nmax <= 1024) return 128;
  return s->nmax > 2048 ? 512 : 256;
}

// the models whose partitioned solve is the chunked one
constexpr bool chunked_model() { return Model::NS <= 8; }

template <int T> void launch_diffuse_chunk(FmsSolver *s, int q, int ie) {
  const size_t lds = (size_t)(20 * (T / 64) + s->nmax) * sizeof(double);
  FMS_LAUNCH(s, (fms::k_diffuse_chunk<T, 8>), dim3(s->F), dim3(T), lds, s->fibers(), s->d_vm, step_ref(s, q), ie);
}

int launch_thomas(FmsSolver *s, int q) {
  KernelTimer timer(s, FMS_KERNEL_DIFFUSION);
  const int ie = s->scheme == FMS_IMPLICIT_EULER;
  if constexpr (chunked_model()) {
    if (s->thomas == FMS_THOMAS_PARTITIONED) {
      const int T = chunk_threads(s);
      if (T == 128) launch_diffuse_chunk<128>(s, q, ie);
      else if (T == 512) launch_diffuse_chunk<512>(s, q, ie);
      else launch_diffuse_chunk<256>(s, q, ie);
      HIP_TRY(hipGetLastError());
      s->n_launch_thomas++;
      return 0;
    }
  }
  if (s->thomas == FMS_THOMAS_SERIAL) {
    if (fms::serial_by_lanes(s->F, s->nmax))
      FMS_LAUNCH(s, fms::k_thomas_serial_lanes, dim3((s->F + 63) / 64), dim3(64), 0, s->fibers(), s->d_vm, s->d_cA,
                 s->d_dA, step_ref(s, q), ie);
    else
      FMS_LAUNCH(s, fms::k_thomas_serial, dim3(s->F), dim3(64), 0, s->fibers(), s->d_vm, s->d_cA, s->d_dA,
                 step_ref(s, q), ie);
  } else if constexpr (!chunked_model()) {
    // rows per chunk: at most ceil(nmax / 256) (>= 3 for fibres under 512 nodes);
    // the smallest register array that holds them
    const size_t lds = (size_t)(fms::pcr_lds_doubles<PART_T>() + s->nmax) * sizeof(double);
    if (s->nmax <= 1024)
      FMS_LAUNCH(s, (fms::k_thomas_part<PART_T, 4>), dim3(s->F), dim3(PART_T), lds, s->fibers(),
                 s->d_vm, step_ref(s, q), ie);
    else if (s->nmax <= 2048)
      FMS_LAUNCH(s, (fms::k_thomas_part<PART_T, 8>), dim3(s->F), dim3(PART_T), lds, s->fibers(),
                 s->d_vm, step_ref(s, q), ie);
    else
      FMS_LAUNCH(s, (fms::k_thomas_part<PART_T, 16>), dim3(s->F), dim3(PART_T), lds, s->fibers(),
                 s->d_vm, step_ref(s, q), ie);
  }
  HIP_TRY(hipGetLastError());
  s->n_launch_thomas++;
  return 0;
}

int launch_spikes(FmsSolver *s, int q) {
  KernelTimer timer(s, FMS_KERNEL_OTHER);
  const int threads = 256;
  const long long blocks = (s->N + threads - 1) / threads;
  FMS_LAUNCH(s, fms::k_spikes, dim3((unsigned)blocks), dim3(threads), 0, s->N, s->d_vm,
             s->d_vprev, s->d_sfirst, s->d_scount, s->spike_th, step_ref(s, q));
  HIP_TRY(hipGetLastError());
  return 0;
}

// one Strang step on the split kernels: reaction half, diffusion, reaction half
// (fast_monodomain_solver_compute.tpp:110-126), step q of the launch sequence
template <class G, class E>
int enqueue_split_step(FmsSolver *s, int q, int n0D, bool store_alg) {
  int rc;
  if ((rc = launch_flags(s, q, 0, n0D))) return rc;
  if ((rc = launch_reaction<G, E>(s, q, 0, n0D, false))) return rc;
  if ((rc = launch_thomas(s, q))) return rc;
  if ((rc = launch_flags(s, q, 1, n0D))) return rc;
  if ((rc = launch_reaction<G, E>(s, q, 1, n0D, store_alg))) return rc;
  if (s->spikes && (rc = launch_spikes(s, q))) return rc;
  return 0;
}

// paired form, between the first half of the call's first step and the second
// half of its last step: the diffusion of step q, then the second half of step
// q and the first half of step q+1 in one launch
template <class G, class E>
int enqueue_pair_body(FmsSolver *s, int q, int n0D) {
  int rc;
  if ((rc = launch_thomas(s, q))) return rc;
  if ((rc = launch_flags_pair(s, q, n0D))) return rc;
  return launch_reaction_pair<G, E>(s, q, n0D);
}

// everything a captured graph of split steps has baked into its kernel arguments
template <class G, class E>
std::vector<unsigned char> graph_signature(const FmsSolver *s, int gsteps, int n0D) {
  const fms::DevFibers fb = s->fibers();
  const fms::DevStim st = s->stim();
  struct {
    const void *vm, *gates, *flags, *cursor, *cA, *dA, *vprev, *sfirst, *scount;
    double vstim, spike_th;
    int spikes, n0D, gsteps, thomas, scheme, nmax, g_is_double, e_is_approx, pair, per_fibre, rthreads,
        cthreads;
  } k;
  memset(&k, 0, sizeof(k));
  k.vm = s->d_vm; k.gates = s->d_gates; k.flags = s->d_flags; k.cursor = s->d_cursor;
  k.cA = s->d_cA; k.dA = s->d_dA; k.vprev = s->d_vprev; k.sfirst = s->d_sfirst; k.scount = s->d_scount;
  k.vstim = s->vstim; k.spike_th = s->spike_th; k.spikes = s->spikes; k.n0D = n0D; k.gsteps = gsteps;
  k.thomas = s->thomas; k.scheme = s->scheme; k.nmax = s->nmax;
  k.pair = s->tune_pair; k.per_fibre = s->tune_reaction_fibre; k.rthreads = s->tune_reaction_threads;
  k.cthreads = chunked_model() && s->thomas == FMS_THOMAS_PARTITIONED ? chunk_threads(s) : 0;
  k.g_is_double = std::is_same<G, double>::value;
  k.e_is_approx = std::is_base_of<fms::ExpApprox, E>::value;
  std::vector<unsigned char> sig(sizeof(fb) + sizeof(st) + sizeof(k));
  memcpy(sig.data(), &fb, sizeof(fb));
  memcpy(sig.data() + sizeof(fb), &st, sizeof(st));
  memcpy(sig.data() + sizeof(fb) + sizeof(st), &k, sizeof(k));
  return sig;
}

void drop_graph(FmsSolver *s) {
  if (s->graph_exec) (void)hipGraphExecDestroy(s->graph_exec);
  s->graph_exec = nullptr;
  s->graph_sig.clear();
}

// capture gsteps split steps (paired: gsteps pair bodies) and the cursor
// advance as one graph
template <class G, class E>
int capture_split_graph(FmsSolver *s, int gsteps, int n0D) {
  drop_graph(s);
  const long long nr = s->n_launch_reaction, nt = s->n_launch_thomas;
  const int prof = s->prof;
  s->prof = 0;   // no timing events inside a captured graph
  HIP_TRY(hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal));
  int rc = 0;
  for (int q = 0; q < gsteps && !rc; q++)
    rc = s->tune_pair ? enqueue_pair_body<G, E>(s, q, n0D) : enqueue_split_step<G, E>(s, q, n0D, false);
  if (!rc) {
    hipLaunchKernelGGL(fms::k_cursor_advance, dim3(1), dim3(64), 0, s->stream, s->d_cursor, gsteps);
    if (hipGetLastError() != hipSuccess) rc = fail(FMS_ERR_HIP, "cursor kernel launch failed during capture");
  }
  hipGraph_t graph = nullptr;
  const hipError_t e = hipStreamEndCapture(s->stream, &graph);
  s->prof = prof;
  s->n_launch_reaction = nr;
  s->n_launch_thomas = nt;
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (e != hipSuccess) return fail(FMS_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
  const hipError_t ei = hipGraphInstantiate(&s->graph_exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (ei != hipSuccess) {
    s->graph_exec = nullptr;
    return fail(FMS_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(ei));
  }
  s->graph_sig = graph_signature<G, E>(s, gsteps, n0D);
  s->n_graph_captures++;
  return 0;
}

// split kernels: K steps, whole groups of tune_graph steps replayed as one
// captured graph, the rest (and a step that returns algebraics) launched eagerly.
// Paired (tune_pair): the first half of step 0, then K-1 bodies (diffusion of
// step q, second half of q + first half of q+1; graphs of tune_graph bodies),
// then the diffusion and second half of step K-1 (which returns algebraics).
template <class G, class E>
int run_split(FmsSolver *s, const double *h_steps, int K, int n0D) {
  int rc;
  if ((rc = upload_steps(s, h_steps, K))) return rc;
  const int gs = s->tune_graph;
  const bool pair = s->tune_pair != 0;
  if (pair) {
    if ((rc = launch_flags(s, 0, 0, n0D))) return rc;
    if ((rc = launch_reaction<G, E>(s, 0, 0, n0D, false))) return rc;
  }
  const int graph_steps_max = pair ? K - 1 : (s->d_alg ? K - 1 : K);
  int done = 0;
  if (gs > 0 && graph_steps_max >= gs) {
    if (s->graph_sig != graph_signature<G, E>(s, gs, n0D) || !s->graph_exec)
      if ((rc = capture_split_graph<G, E>(s, gs, n0D))) return rc;
    const int nrep = graph_steps_max / gs;
    for (int r = 0; r < nrep; r++) HIP_TRY(hipGraphLaunch(s->graph_exec, s->stream));
    done = nrep * gs;
    s->n_launch_reaction += (pair ? 1LL : 2LL) * done;
    s->n_launch_thomas += done;
    s->n_graph_launches += nrep;
  }
  // the cursor now points at row `done`
  if (pair) {
    int q = 0;
    for (; done + q < K - 1; q++)
      if ((rc = enqueue_pair_body<G, E>(s, q, n0D))) return rc;
    if ((rc = launch_thomas(s, q))) return rc;
    if ((rc = launch_flags(s, q, 1, n0D))) return rc;
    if ((rc = launch_reaction<G, E>(s, q, 1, n0D, s->d_alg != nullptr))) return rc;
    if (s->spikes && (rc = launch_spikes(s, q))) return rc;
  } else {
    for (int q = 0; done + q < K; q++)
      if ((rc = enqueue_split_step<G, E>(s, q, n0D, s->d_alg && done + q == K - 1))) return rc;
  }
  s->step_counter += K;
  return 0;
}

template <class G, class E, int T, int NPT, int MMAX>
int launch_fused_npt(FmsSolver *s, const double *d_steps, int K, int n0D, const fms::DevTrace &tr) {
  KernelTimer timer(s, FMS_KERNEL_FUSED);
  const fms::DevSpikes spk = dev_spikes(s);
  int serial = s->thomas == FMS_THOMAS_SERIAL ? fms::SERIAL_PLAIN : 0;
  int red = serial ? 16 * T : fms::pcr_lds_doubles<T>();
  if constexpr (chunked_model()) {
    serial = fms::SERIAL_FACTORED;
    red = fms::serial_lds_doubles(s->nmax);
    if (fms::fused_lds_bytes(red, s->nmax, n0D) > fms::FUSED_LDS_BYTES) {
      serial = fms::SERIAL_PLAIN;
      red = 2 * s->nmax;
    }
  }
  const size_t lds = fms::fused_lds_bytes(red, s->nmax, n0D);
  FMS_LAUNCH(s, (fms::k_fused<Model, G, E, T, MMAX, NPT>), dim3(s->F), dim3(T), lds, s->fibers(), s->stim(),
             s->d_vm, (G *)s->d_gates, d_steps, K, n0D, s->vstim, s->scheme == FMS_IMPLICIT_EULER ? 1 : 0,
             serial, s->d_order, spk, tr);
  HIP_TRY(hipGetLastError());
  s->step_counter += K;
  s->n_launch_fused++;
  return 0;
}

// bytes of the flags that one launch of K steps reads
size_t fibre_flag_bytes(const FmsSolver *s, int K, int n0D) {
  return (size_t)s->F * fms::flag_groups(K, n0D) * sizeof(fms::FlagGroup);
}

// Steps of a launch whose flags need not exceed FIBRE_FLAG_BYTES (or one step): with
// many Heun steps per split step a launch of few steps is long enough, and the flags of
// 512 would take 256 bytes per fibre and Heun step.
constexpr size_t FIBRE_FLAG_BYTES = 64 << 20;
int fibre_launch_steps(const FmsSolver *s, int K, int n0D, size_t bytes) {
  while (K > 1 && (fibre_flag_bytes(s, K, n0D) > bytes || 2LL * K * n0D > (1 << 30))) K = (K + 1) / 2;
  return K;
}

// the flags of K steps, then the steps
template <class G, class E, bool TAPE>
int launch_fibre(FmsSolver *s, const double *d_steps, int K, int n0D, const fms::DevTrace &tr) {
  {
    KernelTimer timer(s, FMS_KERNEL_OTHER);
    FMS_LAUNCH(s, fms::k_fibre_flags, dim3(s->F), dim3(64), 0, s->stim(), d_steps, K, n0D,
               reinterpret_cast<fms::FlagGroup *>(s->d_flags));
    HIP_TRY(hipGetLastError());
  }
  KernelTimer timer(s, FMS_KERNEL_FUSED);
  fms::FibreLaunch l{};
  l.fb = s->fibers();
  l.st = fms::FibreStim{s->stim_mode == FMS_STIM_FIRING_TABLE, s->stim_param, s->vstim, s->d_amp,
                        reinterpret_cast<const fms::FlagGroup *>(s->d_flags)};
  l.vm = s->d_vm;
  l.gates = s->d_gates;
  l.steps = d_steps;
  l.nmax = s->nmax;
  l.K = K;
  l.n0D = n0D;
  l.ie = s->scheme == FMS_IMPLICIT_EULER ? 1 : 0;
  l.order = s->d_order;
  l.spk = dev_spikes(s);
  l.tr = tr;
  l.stream = s->stream;
  if (s->prof_slot >= 0) {
    l.start = s->prof_ev[2 * s->prof_slot];
    l.stop = s->prof_ev[2 * s->prof_slot + 1];
    s->prof_launched = 1;
  }
  fms::fibre_launch<G, E, TAPE>(chunk_threads(s), l);
  HIP_TRY(hipGetLastError());
  s->step_counter += K;
  s->n_launch_fused++;
  return 0;
}

// Resident gates: at most 32 doubles (64 registers) of them per thread beside what the
// reaction and the serial solve need. More, at 8 nodes per thread of an 8-state model,
// left 256 registers, 230 accumulation registers and 390 spilled scalar ones, and that
// build lost the eighth node's states (NaN); streamed gates give the split kernels' bits.
constexpr bool resident_fits(int npt) { return npt * (Model::NS - 1) <= 32; }

// Fused schedules: one workgroup of T threads per fibre; gates resident in
// registers (NPT nodes per thread, small models) or streamed from HBM. The
// partitioned solve needs ceil(n / T) <= MMAX rows per thread, the serial
// solve 2n <= 16 T doubles of LDS scratch (fms_set_tuning checks both).
template <class G, class E>
int launch_fused(FmsSolver *s, const double *d_steps, int K, int n0D, const fms::DevTrace &tr = fms::DevTrace{}) {
  if constexpr (chunked_model() && fms::is_fma<E>::value) {
    // sensors and the tape are the adjoint forward's, which runs in FP64 with any model
    if constexpr (std::is_same<G, double>::value)
      if (tr.sensor_slot || tr.tape) return launch_fibre<G, E, true>(s, d_steps, K, n0D, tr);
    return launch_fibre<G, E, false>(s, d_steps, K, n0D, tr);
  } else {
  const bool resident = s->tune_resident != 0;
  if constexpr (Model::NS <= 8) {
    if (s->tune_threads == 128) {
      // resident gates for at most 8 nodes per thread: 16 per thread spill to
      // scratch, and that build of the fused kernel computed wrong states
      const int npt = (s->nmax + 127) / 128;
      constexpr int NPT = resident_fits(8) ? 8 : 4;
      if (resident && npt <= NPT) return launch_fused_npt<G, E, 128, NPT, 8>(s, d_steps, K, n0D, tr);
      return launch_fused_npt<G, E, 128, 0, 8>(s, d_steps, K, n0D, tr);
    }
  }
  constexpr int T = FUSED_T;
  const int npt = (s->nmax + T - 1) / T;
  if constexpr (Model::NS <= 8) {
    if (resident && npt <= 4) return launch_fused_npt<G, E, T, 4, 8>(s, d_steps, K, n0D, tr);
    if constexpr (resident_fits(8))
      if (resident && npt <= 8) return launch_fused_npt<G, E, T, 8, 8>(s, d_steps, K, n0D, tr);
  }
  // small models come here with the serial solve, of at most 8 rows per thread
  if constexpr (!chunked_model())
    if (npt > 8) return launch_fused_npt<G, E, T, 0, 16>(s, d_steps, K, n0D, tr);
  return launch_fused_npt<G, E, T, 0, 8>(s, d_steps, K, n0D, tr);
  }
}

template <class G, class E>
int run(FmsSolver *s, const double *h_steps, int K, int n0D, bool fused_only);

template <class G, class E>
int run(FmsSolver *s, const double *h_steps, int K, int n0D) {
  // the point-buffer order decides per node: the per-node split kernels. They
  // also take a call without allocation whose flags of one fused step do not fit.
  const bool fibre = chunked_model() && fms::is_fma<E>::value;
  const bool flags_fit = !fibre || !s->noalloc || fibre_flag_bytes(s, 1, n0D) <= s->flags_cap;
  if (s->kernels == FMS_KERNELS_SPLIT || s->vc_width || !flags_fit) {
    if (s->thomas == FMS_THOMAS_SERIAL && !s->d_cA &&
        (dalloc(&s->d_cA, (size_t)s->N) || dalloc(&s->d_dA, (size_t)s->N)))
      return FMS_ERR_HIP;
    return run_split<G, E>(s, h_steps, K, n0D);
  }
  // the fused kernel does not return algebraics: with algebraicsForTransfer
  // requested, the last step of the call runs on the split kernels (same
  // arithmetic, bit-identical states)
  if (s->d_alg) {
    int rc = 0;
    if (K > 1 && (rc = run<G, E>(s, h_steps, K - 1, n0D, true))) return rc;
    if (s->thomas == FMS_THOMAS_SERIAL && !s->d_cA) {
      if (dalloc(&s->d_cA, (size_t)s->N) || dalloc(&s->d_dA, (size_t)s->N)) return FMS_ERR_HIP;
    }
    return run_split<G, E>(s, h_steps + 4 * (size_t)(K - 1), 1, n0D);
  }
  return run<G, E>(s, h_steps, K, n0D, true);
}

template <class G, class E>
int run(FmsSolver *s, const double *h_steps, int K, int n0D, bool fused_only) {
  (void)fused_only;
  // fused: the kernel reads step s+1's record for the first half of step s+1;
  // a launch covers steps [k0, k0+kc) and then finishes the last step itself
  int rc;
  if ((rc = upload_steps(s, h_steps, K, false))) return rc;
  int chunk = s->tune_chunk;
  if constexpr (chunked_model() && fms::is_fma<E>::value) {
    // the flags of a launch: allocated, or as many steps as the fixed scratch holds
    chunk = fibre_launch_steps(s, std::min(chunk, K), n0D, s->noalloc ? s->flags_cap : FIBRE_FLAG_BYTES);
    if (!s->noalloc && ensure_flag_bytes(s, fibre_flag_bytes(s, chunk, n0D))) return FMS_ERR_HIP;
  }
  for (int k0 = 0; k0 < K; k0 += chunk) {
    const int kc = std::min(chunk, K - k0);
    if ((rc = launch_fused<G, E>(s, s->d_steps + 4 * (size_t)k0, kc, n0D))) return rc;
  }
  return 0;
}

// calls fn with the exponential policy of the solver's runs. Runs with the
// partitioned solve of a small model are held to a tolerance and take the fused
// multiply-add forms; the serial solve's runs give the oracle's bits.
template <class Fn> int with_exp(FmsSolver *s, Fn fn) {
  const bool approx = s->exp_mode == FMS_EXP_APPROXIMATE;
  if constexpr (chunked_model()) {
    if (s->thomas == FMS_THOMAS_PARTITIONED) return approx ? fn(fms::ExpApproxFma{}) : fn(fms::ExpLibmFma{});
  }
  return approx ? fn(fms::ExpApprox{}) : fn(fms::ExpLibm{});
}

int dispatch(FmsSolver *s, const double *h_steps, int K, int n0D) {
  if (K <= 0) return 0;
  if (n0D < 1) return fail(FMS_ERR_ARGUMENT, "n0D must be >= 1");
  if (ensure_flags(s, n0D)) return FMS_ERR_HIP;
  return with_exp(s, [&](auto e) {
    using E = decltype(e);
    if (s->precision == FMS_FP64) return run<double, E>(s, h_steps, K, n0D);
    return run<float, E>(s, h_steps, K, n0D);
  });
}

size_t gate_bytes(const FmsSolver *s) { return s->precision == FMS_FP64 ? sizeof(double) : sizeof(float); }

// Device scratch of the allocation-free advance (fms_advance_schedule_noalloc):
// the split-step table and the per-fibre flags of one call. Each GPU the
// library runs on holds its own copy until the process ends; host code uses the
// address hipGetSymbolAddress returns for the current device (noalloc_ptr), never
// the array's name, which in host code is only a stand-in.
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)4 << 20;
constexpr int NOALLOC_MAX_DEVICES = 64;
__device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];
unsigned char *g_noalloc_ptr[NOALLOC_MAX_DEVICES] = {};

// set-up, with the device current: fetch this device's scratch address once
int noalloc_init(int device) {
  if (device < 0 || device >= NOALLOC_MAX_DEVICES) return fail(FMS_ERR_UNSUPPORTED, "device number out of range");
  if (g_noalloc_ptr[device]) return 0;
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr)
    return fail(FMS_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_noalloc_ptr[device] = static_cast<unsigned char *>(ptr);
  return 0;
}

}  // namespace

// ===========================================================================
// C ABI
// ===========================================================================

extern "C" {

int fms_last_error(char *buf, int len) {
  FMS_API_BEGIN
  if (!buf || len <= 0) return FMS_ERR_ARGUMENT;
  snprintf(buf, (size_t)len, "%s", g_last_error.c_str());
  return 0;
  FMS_API_END
}

int fms_model_info(int *n_states, int *n_algebraics, int *n_params, char *name, int name_len) {
  FMS_API_BEGIN
  if (n_states) *n_states = Model::NS;
  if (n_algebraics) *n_algebraics = Model::NA;
  if (n_params) *n_params = Model::NP;
  if (name && name_len > 0) snprintf(name, (size_t)name_len, "%s", Model::name());
  return 0;
  FMS_API_END
}

int fms_model_ops(double *ops_rhs, double *divs_rhs, double *exps_rhs) {
  FMS_API_BEGIN
  if (ops_rhs) *ops_rhs = Model::OPS_RHS;
  if (divs_rhs) *divs_rhs = Model::DIVS_RHS;
  if (exps_rhs) *exps_rhs = Model::EXPS_RHS;
  return 0;
  FMS_API_END
}

int fms_model_defaults(double *states, double *params) {
  FMS_API_BEGIN
  if (states)
    for (int k = 0; k < Model::NS; k++) states[k] = Model::y0(k);
  if (params)
    for (int k = 0; k < Model::NP; k++) params[k] = Model::p0(k);
  return 0;
  FMS_API_END
}

int fms_eval_rhs(const double *states, const double *params, double t, int n, int exp_mode, double *rates,
                 double *algebraics) {
  FMS_API_BEGIN
  if (n <= 0 || !states || !rates || (Model::NP > 0 && !params)) return fail(FMS_ERR_ARGUMENT, "bad arguments");
  if (exp_mode != FMS_EXP_APPROXIMATE && exp_mode != FMS_EXP_LIBM) return fail(FMS_ERR_ARGUMENT, "bad exp_mode");
  const size_t NS = Model::NS, NA = Model::NA, NP = Model::NP > 0 ? Model::NP : 1;
  double *d_y = nullptr, *d_p = nullptr, *d_r = nullptr, *d_a = nullptr;
  int rc = 0;
  if (dalloc(&d_y, NS * n) || dalloc(&d_p, NP * n) || dalloc(&d_r, NS * n) || (algebraics && dalloc(&d_a, NA * n)))
    rc = FMS_ERR_HIP;
  if (!rc && hipMemcpy(d_y, states, NS * n * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) rc = FMS_ERR_HIP;
  if (!rc && Model::NP > 0 && hipMemcpy(d_p, params, NP * n * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
    rc = FMS_ERR_HIP;
  if (!rc) {
    const unsigned blocks = (unsigned)((n + 255) / 256);
    if (exp_mode == FMS_EXP_APPROXIMATE)
      hipLaunchKernelGGL((fms::k_eval_rhs<Model, fms::ExpApprox>), dim3(blocks), dim3(256), 0, 0, d_y, d_p, t, n,
                         d_r, d_a);
    else
      hipLaunchKernelGGL((fms::k_eval_rhs<Model, fms::ExpLibm>), dim3(blocks), dim3(256), 0, 0, d_y, d_p, t, n,
                         d_r, d_a);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) rc = FMS_ERR_HIP;
  }
  if (!rc && hipMemcpy(rates, d_r, NS * n * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess) rc = FMS_ERR_HIP;
  if (!rc && algebraics && hipMemcpy(algebraics, d_a, NA * n * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
    rc = FMS_ERR_HIP;
  for (double *q : {d_y, d_p, d_r, d_a})
    if (q) (void)hipFree(q);
  return rc ? fail(rc, "fms_eval_rhs: device error") : 0;
  FMS_API_END
}

int fms_eval_heun(double *states, const double *params, double t0, double dt, int n_steps, int n, int exp_mode) {
  FMS_API_BEGIN
  if (n <= 0 || n_steps < 0 || !states || (Model::NP > 0 && !params)) return fail(FMS_ERR_ARGUMENT, "bad arguments");
  if (exp_mode != FMS_EXP_APPROXIMATE && exp_mode != FMS_EXP_LIBM) return fail(FMS_ERR_ARGUMENT, "bad exp_mode");
  const size_t NS = Model::NS, NP = Model::NP > 0 ? Model::NP : 1;
  double *d_y = nullptr, *d_p = nullptr;
  int rc = 0;
  if (dalloc(&d_y, NS * n) || dalloc(&d_p, NP * n)) rc = FMS_ERR_HIP;
  if (!rc && hipMemcpy(d_y, states, NS * n * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) rc = FMS_ERR_HIP;
  if (!rc && Model::NP > 0 && hipMemcpy(d_p, params, NP * n * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
    rc = FMS_ERR_HIP;
  if (!rc) {
    const unsigned blocks = (unsigned)((n + 255) / 256);
    if (exp_mode == FMS_EXP_APPROXIMATE)
      hipLaunchKernelGGL((fms::k_eval_heun<Model, fms::ExpApprox>), dim3(blocks), dim3(256), 0, 0, d_y, d_p, t0, dt,
                         n_steps, n);
    else
      hipLaunchKernelGGL((fms::k_eval_heun<Model, fms::ExpLibm>), dim3(blocks), dim3(256), 0, 0, d_y, d_p, t0, dt,
                         n_steps, n);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) rc = FMS_ERR_HIP;
  }
  if (!rc && hipMemcpy(states, d_y, NS * n * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess) rc = FMS_ERR_HIP;
  for (double *q : {d_y, d_p})
    if (q) (void)hipFree(q);
  return rc ? fail(rc, "fms_eval_heun: device error") : 0;
  FMS_API_END
}

// initializeStatesToEquilibrium of the CellML adapter
// (core/src/cellml/03_cellml_adapter.tpp:446-520): classical RK4 on one cell
// with the model's libm functions, the time left at 0 as there, until the
// largest state increment per unit time is below 1e-5; an increment above 1e4
// restarts from the initial values with half the step. The search is one
// serial recurrence run once before the first step, so it runs on the host
// core that calls it (the reference runs it on the host too); the model's
// right-hand side is the same source the device kernels compile.
int fms_equilibrium_states(double *states, const double *params, double dt, long long max_iterations,
                           long long *iterations, double *max_increment, double *dt_out) {
  FMS_API_BEGIN
  if (!states || (Model::NP > 0 && !params) || !(dt > 0) || max_iterations < 0)
    return fail(FMS_ERR_ARGUMENT, "fms_equilibrium_states: bad arguments");
  constexpr int NS = Model::NS;
  fms::FD u[NS], prev[NS], k1[NS], k2[NS], k3[NS], k4[NS], u2[NS], u3[NS], u4[NS], a[Model::NA];
  fms::FD p[Model::NP > 0 ? Model::NP : 1];
  for (int k = 0; k < Model::NP; k++) p[k] = fms::FD(params[k]);
  for (int k = 0; k < NS; k++) u[k] = prev[k] = fms::FD(states[k]);
  const double t = 0.0;
  double incr = 0.0;
  long long it = 0;
  for (; it < max_iterations; it++) {
    Model::template rhs<fms::FD, fms::ExpLibm>(u, p, t, k1, a);
    for (int k = 0; k < NS; k++) u2[k] = fms::FD(u[k].v + dt / 2. * k1[k].v);
    Model::template rhs<fms::FD, fms::ExpLibm>(u2, p, t + dt / 2., k2, a);
    for (int k = 0; k < NS; k++) u3[k] = fms::FD(u[k].v + dt / 2. * k2[k].v);
    Model::template rhs<fms::FD, fms::ExpLibm>(u3, p, t + dt / 2., k3, a);
    for (int k = 0; k < NS; k++) u4[k] = fms::FD(u[k].v + dt * k3[k].v);
    Model::template rhs<fms::FD, fms::ExpLibm>(u4, p, t + dt, k4, a);
    incr = 0.0;
    for (int k = 0; k < NS; k++) {
      const double inc = (k1[k].v + 2 * k2[k].v + 2 * k3[k].v + k4[k].v) / 6.;
      if (std::fabs(inc) > incr) incr = std::fabs(inc);
      u[k] = fms::FD(u[k].v + dt * inc);
    }
    if (incr > 1e4) {
      dt /= 2.0;
      for (int k = 0; k < NS; k++) u[k] = prev[k];
    }
    if (incr < 1e-5) break;
  }
  for (int k = 0; k < NS; k++) states[k] = u[k].v;
  if (iterations) *iterations = it;
  if (max_increment) *max_increment = incr;
  if (dt_out) *dt_out = dt;
  // a state that became NaN never raises the maximum increment (fabs(NaN) > x
  // is false), so the search could stop "converged" on it: report it instead
  for (int k = 0; k < NS; k++)
    if (!std::isfinite(u[k].v))
      return fail(FMS_ERR_STATE, "the equilibrium search reached a non-finite value of state " + std::to_string(k));
  if (!(incr < 1e-5))
    return fail(FMS_ERR_STATE, "equilibrium values of the states were not found within " +
                                   std::to_string(max_iterations) + " RK4 iterations (last increment " +
                                   std::to_string(incr) + ", step " + std::to_string(dt) + ")");
  return 0;
  FMS_API_END
}

int fms_create(const FmsConfig *c, FmsSolver **out) {
  FMS_API_BEGIN
  if (!c || !out) return fail(FMS_ERR_ARGUMENT, "null argument");
  *out = nullptr;
  if (c->n_fibers <= 0 || !c->n_nodes || !c->element_lengths || !c->prefactor)
    return fail(FMS_ERR_ARGUMENT, "n_fibers, n_nodes, element_lengths and prefactor are required");
  if (c->scheme != FMS_IMPLICIT_EULER && c->scheme != FMS_CRANK_NICOLSON)
    return fail(FMS_ERR_ARGUMENT, "scheme must be FMS_IMPLICIT_EULER or FMS_CRANK_NICOLSON");
  if (c->precision != FMS_FP64 && c->precision != FMS_MIXED) return fail(FMS_ERR_ARGUMENT, "bad precision");
  if (c->exp_mode != FMS_EXP_APPROXIMATE && c->exp_mode != FMS_EXP_LIBM) return fail(FMS_ERR_ARGUMENT, "bad exp_mode");
  if (c->thomas != FMS_THOMAS_SERIAL && c->thomas != FMS_THOMAS_PARTITIONED) return fail(FMS_ERR_ARGUMENT, "bad thomas");
  if (c->kernels != FMS_KERNELS_SPLIT && c->kernels != FMS_KERNELS_FUSED) return fail(FMS_ERR_ARGUMENT, "bad kernels");
  FmsSolver *s = new FmsSolver();
  s->F = c->n_fibers;
  s->scheme = c->scheme;
  s->precision = c->precision;
  s->exp_mode = c->exp_mode;
  s->thomas = c->thomas;
  s->kernels = c->kernels;
  s->vstim = c->value_for_stimulated_point;
  s->h_off.resize(s->F + 1);
  s->h_off[0] = 0;
  long long total = 0;
  for (int f = 0; f < s->F; f++) {
    const int n = c->n_nodes[f];
    if (n < 2) {
      delete s;
      return fail(FMS_ERR_ARGUMENT, "every fibre needs at least 2 nodes");
    }
    s->nmax = std::max(s->nmax, n);
    total += n;
    if (total > 0x7fffffffLL) {
      delete s;
      return fail(FMS_ERR_ARGUMENT, "more than 2^31-1 nodes in one solver");
    }
    s->h_off[f + 1] = (int)total;
  }
  s->N = total;
  s->GS = (total + 63) / 64 * 64;
  if (s->nmax > 4096 && (s->thomas == FMS_THOMAS_PARTITIONED || s->kernels == FMS_KERNELS_FUSED)) {
    delete s;
    return fail(FMS_ERR_UNSUPPORTED, "fibres longer than 4096 nodes need thomas=SERIAL and kernels=SPLIT");
  }
  if (s->nmax > 2048 && s->thomas == FMS_THOMAS_SERIAL && s->kernels == FMS_KERNELS_FUSED) {
    // the fused serial solve keeps its two n-long recurrences in the 16*256-double LDS scratch
    delete s;
    return fail(FMS_ERR_UNSUPPORTED, "the fused kernel's serial solve takes fibres of <= 2048 nodes");
  }
  // fibres longest first for the fused kernel (LPT over the dispatcher)
  s->h_order.resize(s->F);
  for (int f = 0; f < s->F; f++) s->h_order[f] = f;
  std::stable_sort(s->h_order.begin(), s->h_order.end(),
                   [&](int a, int b) { return c->n_nodes[a] > c->n_nodes[b]; });

  int rc = 0;
  auto chk = [&](int r) {
    if (r && !rc) rc = r;
  };
  if (hipGetDevice(&s->device) != hipSuccess) {
    delete s;
    return fail(FMS_ERR_HIP, "hipGetDevice failed");
  }
  if (int r = noalloc_init(s->device)) {
    delete s;
    return r;
  }
  if (hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess) {
    delete s;
    return fail(FMS_ERR_HIP, "hipStreamCreate failed");
  }
  const long long N = s->N;
  const int F = s->F;
  chk(dalloc(&s->d_off, F + 1));
  chk(dalloc(&s->d_node_fiber, (size_t)N));
  chk(dalloc(&s->d_sb, F));
  chk(dalloc(&s->d_se, F));
  chk(dalloc(&s->d_order, F));
  chk(dalloc(&s->d_h, (size_t)(N - F)));
  chk(dalloc(&s->d_pf, F));
  chk(dalloc(&s->d_params, (size_t)F * (Model::NP > 0 ? Model::NP : 1)));
  chk(dalloc(&s->d_vm, (size_t)N));
  chk(dalloc(&s->d_hasbeen, (size_t)F));
  chk(dalloc(&s->d_cursor, 4));
  chk(hipMalloc(&s->d_gates, (size_t)(Model::NS - 1) * s->GS * gate_bytes(s) + 8) == hipSuccess ? 0 : FMS_ERR_HIP);
  if (s->thomas == FMS_THOMAS_SERIAL && s->kernels == FMS_KERNELS_SPLIT) {
    chk(dalloc(&s->d_cA, (size_t)N));
    chk(dalloc(&s->d_dA, (size_t)N));
  }
  if (rc) {
    free_all(s);
    delete s;
    return fail(FMS_ERR_HIP, "device allocation failed: " + g_last_error);
  }
  std::vector<int> node_fiber((size_t)N);
  for (int f = 0; f < F; f++)
    for (int i = s->h_off[f]; i < s->h_off[f + 1]; i++) node_fiber[i] = f;
  std::vector<int> zeros(F, 0);
  std::vector<double> params((size_t)F * (Model::NP > 0 ? Model::NP : 1));
  for (int f = 0; f < F; f++)
    for (int k = 0; k < Model::NP; k++)
      params[(size_t)f * Model::NP + k] = c->parameters ? c->parameters[(size_t)f * Model::NP + k] : Model::p0(k);
  chk(h2d(s->d_off, s->h_off.data(), F + 1, s->stream));
  chk(h2d(s->d_node_fiber, node_fiber.data(), (size_t)N, s->stream));
  chk(h2d(s->d_sb, zeros.data(), F, s->stream));
  chk(h2d(s->d_se, zeros.data(), F, s->stream));
  chk(h2d(s->d_order, s->h_order.data(), F, s->stream));
  if (!rc && hipMemsetAsync(s->d_hasbeen, 0, F, s->stream) != hipSuccess) rc = FMS_ERR_HIP;
  chk(h2d(s->d_h, c->element_lengths, (size_t)(N - F), s->stream));
  chk(h2d(s->d_pf, c->prefactor, F, s->stream));
  chk(h2d(s->d_params, params.data(), params.size(), s->stream));
  // initial states, state-major
  std::vector<double> y0(Model::NS);
  for (int k = 0; k < Model::NS; k++) y0[k] = c->initial_states ? c->initial_states[k] : Model::y0(k);
  {
    std::vector<double> v((size_t)N, y0[0]);
    chk(h2d(s->d_vm, v.data(), (size_t)N, s->stream));
    if (s->precision == FMS_FP64) {
      std::vector<double> g((size_t)(Model::NS - 1) * s->GS, 0.0);
      for (int k = 1; k < Model::NS; k++)
        std::fill(g.begin() + (size_t)(k - 1) * s->GS, g.begin() + (size_t)(k - 1) * s->GS + N, y0[k]);
      chk(h2d((double *)s->d_gates, g.data(), g.size(), s->stream));
    } else {
      std::vector<float> g((size_t)(Model::NS - 1) * s->GS, 0.0f);
      for (int k = 1; k < Model::NS; k++)
        std::fill(g.begin() + (size_t)(k - 1) * s->GS, g.begin() + (size_t)(k - 1) * s->GS + N, (float)y0[k]);
      chk(h2d((float *)s->d_gates, g.data(), g.size(), s->stream));
    }
  }
  if (!rc && hipStreamSynchronize(s->stream) != hipSuccess) rc = fail(FMS_ERR_HIP, "upload failed");
  if (rc) {
    free_all(s);
    delete s;
    return rc;
  }
  *out = s;
  return 0;
  FMS_API_END
}

int fms_destroy(FmsSolver *s) {
  FMS_API_BEGIN
  if (!s) return 0;
  if (s->stream) (void)hipStreamSynchronize(s->stream);
  free_all(s);
  delete s;
  return 0;
  FMS_API_END
}

int fms_set_stimulation(FmsSolver *s, const FmsStimulation *st) {
  FMS_API_BEGIN
  if (!s || !st) return fail(FMS_ERR_ARGUMENT, "null argument");
  const int F = s->F;
  if (st->mode == FMS_STIM_NONE) {
    s->stim_mode = FMS_STIM_NONE;
    return 0;
  }
  if (!st->stim_begin || !st->stim_end) return fail(FMS_ERR_ARGUMENT, "stim_begin/stim_end required");
  int rc = 0;
  auto chk = [&](int r) {
    if (r && !rc) rc = r;
  };
  chk(h2d(s->d_sb, st->stim_begin, F, s->stream));
  chk(h2d(s->d_se, st->stim_end, F, s->stream));
  if (st->mode == FMS_STIM_FIRING_TABLE) {
    if (st->firing_rows <= 0 || st->firing_cols <= 0 || !st->firing_events || !st->motor_unit ||
        !st->call_frequency || !st->repeat_after_first_call || !st->call_enable_begin || !st->jitter_offset ||
        !st->jitter_count)
      return fail(FMS_ERR_ARGUMENT, "firing-table stimulation needs the table and per-fibre settings");
    int njit = 0;
    for (int f = 0; f < F; f++) njit = std::max(njit, st->jitter_offset[f] + st->jitter_count[f]);
    s->fe_rows = st->firing_rows;
    s->fe_cols = st->firing_cols;
    const size_t nfe = (size_t)st->firing_rows * st->firing_cols;
    if (!s->d_fe) {
      chk(dalloc(&s->d_mu, F)); chk(dalloc(&s->d_joff, F)); chk(dalloc(&s->d_jcnt, F)); chk(dalloc(&s->d_jidx, F));
      chk(dalloc(&s->d_freq, F)); chk(dalloc(&s->d_rep, F)); chk(dalloc(&s->d_beg, F)); chk(dalloc(&s->d_last, F));
      chk(dalloc(&s->d_curjit, F)); chk(dalloc(&s->d_curr, F));
      chk(dalloc(&s->d_log_count, 1));
    } else {
      HIP_TRY(hipFree(s->d_fe));
      if (s->d_jit) HIP_TRY(hipFree(s->d_jit));
      s->d_jit = nullptr;
    }
    chk(dalloc(&s->d_fe, nfe));
    chk(dalloc(&s->d_jit, (size_t)std::max(njit, 1)));
    if (rc) return rc;
    chk(h2d(s->d_fe, st->firing_events, nfe, s->stream));
    chk(h2d(s->d_mu, st->motor_unit, F, s->stream));
    chk(h2d(s->d_freq, st->call_frequency, F, s->stream));
    chk(h2d(s->d_rep, st->repeat_after_first_call, F, s->stream));
    chk(h2d(s->d_beg, st->call_enable_begin, F, s->stream));
    if (njit > 0 && st->jitter) chk(h2d(s->d_jit, st->jitter, (size_t)njit, s->stream));
    chk(h2d(s->d_joff, st->jitter_offset, F, s->stream));
    chk(h2d(s->d_jcnt, st->jitter_count, F, s->stream));
    // lastStimulationCheckTime = enableBegin - 1e-13 - 1/(f + 0)
    // (fast_monodomain_solver_initialization.tpp:342-344)
    std::vector<double> last(F);
    for (int f = 0; f < F; f++)
      last[f] = st->last_check_time ? st->last_check_time[f]
                                    : st->call_enable_begin[f] - 1e-13 - 1. / (st->call_frequency[f] + 0.0);
    chk(h2d(s->d_last, last.data(), F, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_curjit, 0, F * sizeof(double), s->stream));
    HIP_TRY(hipMemsetAsync(s->d_jidx, 0, F * sizeof(int), s->stream));
    HIP_TRY(hipMemsetAsync(s->d_curr, 0, F, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_hasbeen, 0, F, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_log_count, 0, sizeof(int), s->stream));
    if (st->log_capacity > 0) {
      if (s->d_log_time) HIP_TRY(hipFree(s->d_log_time));
      if (s->d_log_fiber) HIP_TRY(hipFree(s->d_log_fiber));
      chk(dalloc(&s->d_log_time, (size_t)st->log_capacity));
      chk(dalloc(&s->d_log_fiber, (size_t)st->log_capacity));
    }
    s->log_cap = st->log_capacity;
  } else if (st->mode == FMS_STIM_CURRENT) {
    if (!st->onset || !st->duration || !st->amplitude) return fail(FMS_ERR_ARGUMENT, "current pulses need onset/duration/amplitude");
    if (st->stim_param < 0 || st->stim_param >= Model::NP) return fail(FMS_ERR_ARGUMENT, "stim_param out of range");
    if (!s->d_onset) {
      chk(dalloc(&s->d_onset, F)); chk(dalloc(&s->d_dur, F)); chk(dalloc(&s->d_amp, F));
    }
    if (rc) return rc;
    chk(h2d(s->d_onset, st->onset, F, s->stream));
    chk(h2d(s->d_dur, st->duration, F, s->stream));
    chk(h2d(s->d_amp, st->amplitude, F, s->stream));
    s->stim_param = st->stim_param;
  } else {
    return fail(FMS_ERR_ARGUMENT, "unknown stimulation mode");
  }
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(s->stream));
  s->stim_mode = st->mode;
  return 0;
  FMS_API_END
}

int fms_advance(FmsSolver *s, double t0, double dts, int n_split, double dt0D, int n0D, double dt1D, int n1D) {
  FMS_API_BEGIN
  (void)n1D;
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  if (n_split <= 0) return 0;
  std::vector<double> tab(4 * (size_t)n_split);
  for (int k = 0; k < n_split; k++) {
    tab[4 * (size_t)k] = t0 + k * dts;   // currentTime = startTime + timeStepNo*timeStepWidthSplitting
    tab[4 * (size_t)k + 1] = dts;
    tab[4 * (size_t)k + 2] = dt0D;
    tab[4 * (size_t)k + 3] = dt1D;
  }
  return dispatch(s, tab.data(), n_split, n0D);
  FMS_API_END
}

int fms_advance_schedule(FmsSolver *s, const double *steps, int n_steps, int n0D) {
  FMS_API_BEGIN
  if (!s || (!steps && n_steps > 0)) return fail(FMS_ERR_ARGUMENT, "null argument");
  return dispatch(s, steps, n_steps, n0D);
  FMS_API_END
}

int fms_advance_schedule_noalloc(FmsSolver *s, const double *steps, int n_steps, int n0D) {
  FMS_API_BEGIN
  if (!s || (!steps && n_steps > 0)) return fail(FMS_ERR_ARGUMENT, "null argument");
  if (n_steps <= 0) return 0;
  if (n0D < 1) return fail(FMS_ERR_ARGUMENT, "n0D must be >= 1");
  unsigned char *base = s->device >= 0 && s->device < NOALLOC_MAX_DEVICES ? g_noalloc_ptr[s->device] : nullptr;
  if (!base) return fail(FMS_ERR_STATE, "no scratch address for the solver's device");
  // the table (n_steps + 1 records of 4 doubles) and the flags (2 F n0D bytes)
  const size_t table_bytes = ((size_t)(n_steps + 1) * 4 * sizeof(double) + 255) / 256 * 256;
  const size_t flag_bytes = (size_t)2 * s->F * n0D;
  if (table_bytes + flag_bytes > NOALLOC_SCRATCH_BYTES)
    return fail(FMS_ERR_UNSUPPORTED,
                "fms_advance_schedule_noalloc: " + std::to_string(n_steps) + " steps of " + std::to_string(s->F) +
                    " fibres need " + std::to_string(table_bytes + flag_bytes) + " bytes of scratch, more than the " +
                    std::to_string(NOALLOC_SCRATCH_BYTES) + " bytes it has (32 bytes per step plus 2 bytes per "
                    "fibre and Heun step); split the call");
  // schedules that would allocate are refused: the serial solve's scratch is
  // made at fms_create only for the split kernels
  const bool split_path = s->kernels == FMS_KERNELS_SPLIT || s->vc_width || s->d_alg;
  if (s->thomas == FMS_THOMAS_SERIAL && split_path && !s->d_cA)
    return fail(FMS_ERR_UNSUPPORTED, "fms_advance_schedule_noalloc: this schedule needs the serial solve's scratch; "
                                     "call fms_advance_schedule once first");
  double *keep_steps = s->d_steps;
  unsigned char *keep_flags = s->d_flags;
  const int keep_steps_cap = s->steps_cap, keep_graph = s->tune_graph;
  const size_t keep_flags_cap = s->flags_cap;
  s->d_steps = reinterpret_cast<double *>(base);
  s->steps_cap = (int)(table_bytes / sizeof(double));
  s->d_flags = base + table_bytes;
  s->flags_cap = NOALLOC_SCRATCH_BYTES - table_bytes;
  s->tune_graph = 0;   // a graph capture would allocate: eager launches
  s->noalloc = true;
  const int rc = dispatch(s, steps, n_steps, n0D);
  s->noalloc = false;
  s->d_steps = keep_steps;
  s->d_flags = keep_flags;
  s->steps_cap = keep_steps_cap;
  s->flags_cap = keep_flags_cap;
  s->tune_graph = keep_graph;
  if (rc) {
    (void)hipStreamSynchronize(s->stream);
    return rc;
  }
  // return once the kernels are done with the scratch, so that calls made one
  // after another on this device never overlap
  HIP_TRY(hipStreamSynchronize(s->stream));
  return 0;
  FMS_API_END
}

int fms_synchronize(FmsSolver *s) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  HIP_TRY(hipStreamSynchronize(s->stream));
  return 0;
  FMS_API_END
}

int fms_total_nodes(FmsSolver *s, long long *n) {
  FMS_API_BEGIN
  if (!s || !n) return fail(FMS_ERR_ARGUMENT, "null argument");
  *n = s->N;
  return 0;
  FMS_API_END
}

int fms_get_states(FmsSolver *s, int k, double *out) {
  FMS_API_BEGIN
  if (!s || !out) return fail(FMS_ERR_ARGUMENT, "null argument");
  if (k < 0 || k >= Model::NS) return fail(FMS_ERR_ARGUMENT, "state index out of range");
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (k == 0) {
    HIP_TRY(hipMemcpy(out, s->d_vm, (size_t)s->N * sizeof(double), hipMemcpyDeviceToHost));
  } else if (s->precision == FMS_FP64) {
    HIP_TRY(hipMemcpy(out, (double *)s->d_gates + (size_t)(k - 1) * s->GS, (size_t)s->N * sizeof(double),
                      hipMemcpyDeviceToHost));
  } else {
    std::vector<float> tmp((size_t)s->N);
    HIP_TRY(hipMemcpy(tmp.data(), (float *)s->d_gates + (size_t)(k - 1) * s->GS, (size_t)s->N * sizeof(float),
                      hipMemcpyDeviceToHost));
    for (long long i = 0; i < s->N; i++) out[i] = tmp[(size_t)i];
  }
  return 0;
  FMS_API_END
}

int fms_set_states(FmsSolver *s, int k, const double *in) {
  FMS_API_BEGIN
  if (!s || !in) return fail(FMS_ERR_ARGUMENT, "null argument");
  if (k < 0 || k >= Model::NS) return fail(FMS_ERR_ARGUMENT, "state index out of range");
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (k == 0) {
    HIP_TRY(hipMemcpy(s->d_vm, in, (size_t)s->N * sizeof(double), hipMemcpyHostToDevice));
  } else if (s->precision == FMS_FP64) {
    HIP_TRY(hipMemcpy((double *)s->d_gates + (size_t)(k - 1) * s->GS, in, (size_t)s->N * sizeof(double),
                      hipMemcpyHostToDevice));
  } else {
    std::vector<float> tmp((size_t)s->N);
    for (long long i = 0; i < s->N; i++) tmp[(size_t)i] = (float)in[i];
    HIP_TRY(hipMemcpy((float *)s->d_gates + (size_t)(k - 1) * s->GS, tmp.data(), (size_t)s->N * sizeof(float),
                      hipMemcpyHostToDevice));
  }
  return 0;
  FMS_API_END
}

int fms_set_algebraics_for_transfer(FmsSolver *s, const int *idx, int count) {
  FMS_API_BEGIN
  if (!s || count < 0 || (count > 0 && !idx)) return fail(FMS_ERR_ARGUMENT, "bad argument");
  for (int k = 0; k < count; k++)
    if (idx[k] < 0 || idx[k] >= Model::NA) return fail(FMS_ERR_ARGUMENT, "algebraic index out of range");
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (s->d_alg_idx) HIP_TRY(hipFree(s->d_alg_idx));
  if (s->d_alg) HIP_TRY(hipFree(s->d_alg));
  s->d_alg_idx = nullptr;
  s->d_alg = nullptr;
  s->n_alg_idx = count;
  if (count == 0) return 0;
  if (dalloc(&s->d_alg_idx, (size_t)count) || dalloc(&s->d_alg, (size_t)count * s->N)) return FMS_ERR_HIP;
  HIP_TRY(hipMemcpy(s->d_alg_idx, idx, count * sizeof(int), hipMemcpyHostToDevice));
  HIP_TRY(hipMemset(s->d_alg, 0, (size_t)count * s->N * sizeof(double)));
  return 0;
  FMS_API_END
}

int fms_get_algebraics(FmsSolver *s, double *out) {
  FMS_API_BEGIN
  if (!s || !out) return fail(FMS_ERR_ARGUMENT, "null argument");
  if (!s->d_alg) return fail(FMS_ERR_STATE, "no algebraics for transfer configured");
  HIP_TRY(hipStreamSynchronize(s->stream));
  HIP_TRY(hipMemcpy(out, s->d_alg, (size_t)s->n_alg_idx * s->N * sizeof(double), hipMemcpyDeviceToHost));
  return 0;
  FMS_API_END
}

int fms_enable_spike_detection(FmsSolver *s, double th) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (!s->d_vprev) {
    if (dalloc(&s->d_vprev, (size_t)s->N) || dalloc(&s->d_sfirst, (size_t)s->N) || dalloc(&s->d_scount, (size_t)s->N))
      return FMS_ERR_HIP;
  }
  HIP_TRY(hipMemcpy(s->d_vprev, s->d_vm, (size_t)s->N * sizeof(double), hipMemcpyDeviceToDevice));
  std::vector<int> m1((size_t)s->N, -1);
  HIP_TRY(hipMemcpy(s->d_sfirst, m1.data(), (size_t)s->N * sizeof(int), hipMemcpyHostToDevice));
  HIP_TRY(hipMemset(s->d_scount, 0, (size_t)s->N * sizeof(int)));
  s->spikes = 1;
  s->spike_th = th;
  return 0;
  FMS_API_END
}

int fms_get_spikes(FmsSolver *s, int *first, int *count) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  if (!s->spikes) return fail(FMS_ERR_STATE, "spike detection is not enabled");
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (first) HIP_TRY(hipMemcpy(first, s->d_sfirst, (size_t)s->N * sizeof(int), hipMemcpyDeviceToHost));
  if (count) HIP_TRY(hipMemcpy(count, s->d_scount, (size_t)s->N * sizeof(int), hipMemcpyDeviceToHost));
  return 0;
  FMS_API_END
}

int fms_get_stimulation_log(FmsSolver *s, int *count, double *times, int *fibers, int cap) {
  FMS_API_BEGIN
  if (!s || !count) return fail(FMS_ERR_ARGUMENT, "null argument");
  *count = 0;
  if (s->stim_mode != FMS_STIM_FIRING_TABLE || s->log_cap <= 0) return 0;
  HIP_TRY(hipStreamSynchronize(s->stream));
  HIP_TRY(hipMemcpy(count, s->d_log_count, sizeof(int), hipMemcpyDeviceToHost));
  const int n = std::min(std::min(*count, s->log_cap), cap);
  if (n > 0 && times) HIP_TRY(hipMemcpy(times, s->d_log_time, n * sizeof(double), hipMemcpyDeviceToHost));
  if (n > 0 && fibers) HIP_TRY(hipMemcpy(fibers, s->d_log_fiber, n * sizeof(int), hipMemcpyDeviceToHost));
  return 0;
  FMS_API_END
}

int fms_set_tuning(FmsSolver *s, int key, int value) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  switch (key) {
    case FMS_TUNE_STEPS_PER_LAUNCH:
      if (value < 1) return fail(FMS_ERR_ARGUMENT, "steps per launch must be >= 1");
      s->tune_chunk = value;
      return 0;
    case FMS_TUNE_ONLY_IF_STIMULATED:
      if (value < 0 || value > 1) return fail(FMS_ERR_ARGUMENT, "onlyComputeIfHasBeenStimulated is 0 or 1");
      s->only_if_stimulated = value;
      return 0;
    case FMS_TUNE_RESIDENT_GATES:
      if (value < -1 || value > 1) return fail(FMS_ERR_ARGUMENT, "resident must be -1, 0 or 1");
      if (value == 1 && (s->nmax > 8 * s->tune_threads || Model::NS > 8))
        return fail(FMS_ERR_UNSUPPORTED, "resident gates need <= 8 nodes per thread and <= 8 states");
      s->tune_resident = value;
      return 0;
    case FMS_TUNE_THREADS:
      if (value != 128 && value != 256) return fail(FMS_ERR_ARGUMENT, "threads per fibre must be 128 or 256");
      if (value == 128) {
        if (Model::NS > 8) return fail(FMS_ERR_UNSUPPORTED, "128 threads per fibre are built for models of <= 8 states");
        if (s->tune_resident == 1 && s->nmax > 1024)
          return fail(FMS_ERR_UNSUPPORTED, "resident gates with 128 threads per fibre need fibres of <= 1024 nodes");
        if (s->nmax > 2048) return fail(FMS_ERR_UNSUPPORTED, "128 threads per fibre need fibres of <= 2048 nodes");
        if (s->thomas == FMS_THOMAS_SERIAL && s->nmax > 1024)
          return fail(FMS_ERR_UNSUPPORTED, "128 threads per fibre with the serial solve need fibres of <= 1024 nodes");
      }
      s->tune_threads = value;
      return 0;
    case FMS_TUNE_GRAPH_STEPS:
      if (value < 0 || value > 4096) return fail(FMS_ERR_ARGUMENT, "graph steps must be 0..4096");
      s->tune_graph = value;
      return 0;
    case FMS_TUNE_REACTION_PER_FIBRE:
      if (value < 0 || value > 1) return fail(FMS_ERR_ARGUMENT, "reaction per fibre is 0 or 1");
      s->tune_reaction_fibre = value;
      return 0;
    case FMS_TUNE_REACTION_THREADS:
      if (value != 64 && value != 256) return fail(FMS_ERR_ARGUMENT, "reaction threads per fibre are 64 or 256");
      s->tune_reaction_threads = value;
      return 0;
    case FMS_TUNE_PAIR_HALVES:
      if (value < 0 || value > 1) return fail(FMS_ERR_ARGUMENT, "paired reaction halves is 0 or 1");
      s->tune_pair = value;
      return 0;
    case FMS_TUNE_ADJOINT:
      if (value < FMS_ADJOINT_OVERLAP || value > FMS_ADJOINT_OVERLAP_RECOMPUTE_PRIORITY)
        return fail(FMS_ERR_ARGUMENT, "adjoint schedule is FMS_ADJOINT_OVERLAP, _OVERLAP_PRIORITY, _SERIAL or "
                                      "_OVERLAP_RECOMPUTE_PRIORITY");
      s->tune_adjoint = value;
      return 0;
    case FMS_TUNE_ADJOINT_THREADS:
      if (value != 256 && value != 512 && value != 1024)
        return fail(FMS_ERR_ARGUMENT, "adjoint threads per fibre are 256, 512 or 1024");
      if (value > 256 && s->nmax > 2048 * value / 1024)
        return fail(FMS_ERR_UNSUPPORTED, "512 (1024) adjoint threads per fibre take fibres of <= 2048 nodes");
      s->tune_adjoint_threads = value;
      return 0;
    case FMS_TUNE_ADJOINT_TAPE:
      if (value < FMS_ADJOINT_TAPE_AUTO || value > FMS_ADJOINT_TAPE_WHOLE)
        return fail(FMS_ERR_ARGUMENT, "adjoint tape is FMS_ADJOINT_TAPE_AUTO, _SEGMENTS or _WHOLE");
      s->tune_adjoint_tape = value;
      return 0;
    case FMS_TUNE_PROFILE_KERNELS:
      if (value < 0 || value > 1) return fail(FMS_ERR_ARGUMENT, "kernel profiling is 0 or 1");
      for (hipEvent_t &e : s->prof_ev)
        if (value && !e) HIP_TRY(hipEventCreate(&e));
      if (!value) prof_drain(s);
      s->prof = value;
      return 0;
    default:
      return fail(FMS_ERR_ARGUMENT, "unknown tuning key");
  }
  FMS_API_END
}

int fms_set_point_buffer_order(FmsSolver *s, int width, const int *nmj) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  if (width < 0 || width > 64) return fail(FMS_ERR_ARGUMENT, "point-buffer width must be 0..64");
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (width == 0) {
    s->vc_width = 0;
    return 0;
  }
  if (!nmj) return fail(FMS_ERR_ARGUMENT, "the point-buffer order needs each fibre's stimulation point");
  // centre buffer of each fibre as the sweep finds it (compute.tpp:158-166):
  // buffer b belongs to fibre floor(b * W / n_0) and is its centre if
  // (unsigned long)(nmj - (b*W - offset)) < W
  const int F = s->F;
  const long long nbuf = (s->N + width - 1) / width;
  const double factor = (double)width / (s->h_off[1] - s->h_off[0]);
  std::vector<int> centre(F, -1);
  for (long long b = 0; b < nbuf; b++) {
    int fb = (int)((double)b * factor);
    fb = std::min(std::max(fb, 0), F - 1);
    const long long index_in_fibre = b * width - s->h_off[fb];
    if ((unsigned long)((long long)nmj[fb] - index_in_fibre) < (unsigned long)width) {
      if (b > 0x7fffffffLL) return fail(FMS_ERR_UNSUPPORTED, "too many point buffers");
      centre[fb] = (int)b;
    }
  }
  if (!s->d_vc_centre && dalloc(&s->d_vc_centre, (size_t)F)) return FMS_ERR_HIP;
  HIP_TRY(hipMemcpy(s->d_vc_centre, centre.data(), F * sizeof(int), hipMemcpyHostToDevice));
  s->vc_width = width;
  s->vc_factor = factor;
  return 0;
  FMS_API_END
}

int fms_record_event(FmsSolver *s, int slot) {
  FMS_API_BEGIN
  if (!s || slot < 0 || slot >= 8) return fail(FMS_ERR_ARGUMENT, "event slot must be 0..7");
  if (!s->events[slot]) HIP_TRY(hipEventCreate(&s->events[slot]));
  HIP_TRY(hipEventRecord(s->events[slot], s->stream));
  return 0;
  FMS_API_END
}

int fms_event_elapsed_ms(FmsSolver *s, int from, int to, double *ms) {
  FMS_API_BEGIN
  if (!s || !ms || from < 0 || from >= 8 || to < 0 || to >= 8 || !s->events[from] || !s->events[to])
    return fail(FMS_ERR_ARGUMENT, "events not recorded");
  HIP_TRY(hipEventSynchronize(s->events[to]));
  float f = 0.f;
  HIP_TRY(hipEventElapsedTime(&f, s->events[from], s->events[to]));
  *ms = f;
  return 0;
  FMS_API_END
}

int fms_kernel_times(FmsSolver *s, double *ms, long long *launches, int reset) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  prof_drain(s);
  for (int k = 0; k < FMS_KERNEL_CLASSES; k++) {
    if (ms) ms[k] = s->prof_ms[k];
    if (launches) launches[k] = s->prof_n[k];
    if (reset) {
      s->prof_ms[k] = 0;
      s->prof_n[k] = 0;
    }
  }
  return 0;
  FMS_API_END
}

int fms_graph_counts(FmsSolver *s, long long *captures, long long *replays) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  if (captures) *captures = s->n_graph_captures;
  if (replays) *replays = s->n_graph_launches;
  return 0;
  FMS_API_END
}

int fms_launch_counts(FmsSolver *s, long long *fused, long long *reaction, long long *thomas) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  if (fused) *fused = s->n_launch_fused;
  if (reaction) *reaction = s->n_launch_reaction;
  if (thomas) *thomas = s->n_launch_thomas;
  return 0;
  FMS_API_END
}

}  // extern "C"

#include "fms_schedule.h"
#include "fms_reference_abi.h"

// ===========================================================================
// parameters, sensors and the discrete adjoint
// ===========================================================================
namespace {

template <class T> int ensure(T **p, long long &cap, long long n) {
  if (cap >= n && *p) return 0;
  if (*p) HIP_TRY(hipFree(*p));
  *p = nullptr;
  cap = 0;
  if (dalloc(p, (size_t)n)) return FMS_ERR_HIP;
  cap = n;
  return 0;
}

// one checkpoint: Vm (N doubles) then the gate arrays with their stride
size_t ckpt_doubles(const FmsSolver *s) { return (size_t)s->N + (size_t)(Model::NS - 1) * s->GS; }

int copy_state(FmsSolver *s, double *dst, bool to_ckpt) {
  const size_t n = (size_t)s->N;
  const size_t gb = (size_t)(Model::NS - 1) * s->GS * sizeof(double);
  if (to_ckpt) {
    HIP_TRY(hipMemcpyAsync(dst, s->d_vm, n * sizeof(double), hipMemcpyDeviceToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(dst + n, s->d_gates, gb, hipMemcpyDeviceToDevice, s->stream));
  } else {
    HIP_TRY(hipMemcpyAsync(s->d_vm, dst, n * sizeof(double), hipMemcpyDeviceToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_gates, dst + n, gb, hipMemcpyDeviceToDevice, s->stream));
  }
  return 0;
}

// reverse sweep over all segments; d_dtraces is device memory in the traces'
// layout; leaves dL/d(gNa, gK, gL) in s->d_grad [F][3] and dL/dprefactor in
// s->d_pfbar [F], enqueued on the solver's stream
template <class E> int adjoint_backward_core(FmsSolver *s, const double *d_dtraces) {
  if constexpr (!std::is_same<Model, fms::ModelHH>::value) {
    (void)s; (void)d_dtraces;
    return fail(FMS_ERR_UNSUPPORTED, "the adjoint is implemented for the Hodgkin-Huxley model");
  } else {
    const long long N = s->N;
    const int F = s->F, S = s->n_sensors, K = s->adj_K, Kc = s->adj_interval, n0D = s->adj_n0D;
    const int ie = s->scheme == FMS_IMPLICIT_EULER;
    int rc;
    // at most 4 nodes per thread; 1024 threads would leave 128 registers each
    const int T = s->tune_adjoint_threads == 256 && s->nmax <= 1024 ? 256 : 512;
    long long c1 = 0, c2 = 0, c3 = 0, c4 = 0;
    if ((rc = ensure(&s->d_lam, c1, 4 * N)) || (rc = ensure(&s->d_gacc, c2, 4LL * F * T)) ||
        (rc = ensure(&s->d_pfbar, c3, F)) || (rc = ensure(&s->d_grad, c4, 3 * (long long)F)))
      return rc;
    HIP_TRY(hipMemsetAsync(s->d_lam, 0, 4 * N * sizeof(double), s->stream));
    HIP_TRY(hipMemsetAsync(s->d_gacc, 0, 4LL * F * T * sizeof(double), s->stream));
    // the whole forward's tape (segment seg at seg * tape_len), or two segment
    // buffers: the recompute of segment seg-1 (stream2) runs beside the reverse
    // of segment seg (stream)
    const bool whole = s->adj_whole != 0;
    // segments of Kc steps (checkpoints), or of the solver's steps per fused
    // launch (whole tape: step k's entries at k * step_len)
    const int L = whole ? s->tune_chunk : Kc;
    const size_t step_len = (size_t)(2 * Model::NS + 1) * N;
    const size_t tape_len = (size_t)Kc * step_len;
    const int nseg = (int)((K + (long long)L - 1) / L);
    if (whole && s->tape_cap < (long long)K * (long long)step_len)
      return fail(FMS_ERR_STATE, "the adjoint forward's tape is gone; run fms_adjoint_forward again");
    if (!whole && (rc = ensure(&s->d_tape, s->tape_cap, 2 * (long long)tape_len))) return rc;
    if ((rc = upload_steps(s, s->adj_steps.data(), K, false))) return rc;
    if (!whole && ensure_flag_bytes(s, fibre_flag_bytes(s, std::min(L, K), n0D))) return FMS_ERR_HIP;
    if (!whole) {
      if (!s->stream2 && hipStreamCreateWithFlags(&s->stream2, hipStreamNonBlocking) != hipSuccess)
        return fail(FMS_ERR_HIP, "hipStreamCreate failed");
      for (hipEvent_t &e : s->adj_ev)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
          return fail(FMS_ERR_HIP, "hipEventCreate failed");
      // the recompute stream starts after everything enqueued so far (step table, clears)
      HIP_TRY(hipEventRecord(s->adj_ev[2], s->stream));
      HIP_TRY(hipStreamWaitEvent(s->stream2, s->adj_ev[2], 0));
    }
    const int saved_spikes = s->spikes;
    s->spikes = 0;
    // the serial solve's recompute beside the reverse sweep streams its gates: the
    // resident-gate kernel's registers (194 per lane for HH) do not fit on a SIMD
    // beside a reverse wave, the streamed kernel's (126) do; both give the same
    // bits. The partitioned solve's kernel keeps its gates and ignores the switch.
    const int saved_resident = s->tune_resident;
    if (s->tune_adjoint != FMS_ADJOINT_SERIAL) s->tune_resident = 0;
    hipStream_t main_stream = s->stream;
    for (int idx = 0, seg = nseg - 1; seg >= 0; seg--, idx++) {
      const int k0 = seg * L, kc = std::min(L, K - k0);
      const int buf = idx & 1;
      double *tape = s->d_tape + (whole ? (size_t)k0 * step_len : (size_t)buf * tape_len);
      if (!whole) {
        // recompute the segment from its checkpoint on stream2, recording the tape;
        // the buffer was last read by the reverse of segment seg+2 (serialised
        // schedule: on the solver's own stream, before the reverse sweep)
        if (s->tune_adjoint != FMS_ADJOINT_SERIAL) s->stream = s->stream2;
        if (idx >= 2 && hipStreamWaitEvent(s->stream2, s->adj_ev[buf], 0) != hipSuccess)
          rc = fail(FMS_ERR_HIP, "hipStreamWaitEvent failed");
        if (!rc) rc = copy_state(s, s->d_ckpt + (size_t)seg * ckpt_doubles(s), false);
        fms::DevTrace tr{};
        tr.tape = tape;
        tr.raise_priority = s->tune_adjoint == FMS_ADJOINT_OVERLAP_RECOMPUTE_PRIORITY;
        const long long save = s->step_counter;
        // the forward's kernels, so that the recomputed tape has the forward's bits
        if (!rc)
          rc = with_exp(s, [&](auto e) {
            return launch_fused<double, decltype(e)>(s, s->d_steps + 4 * (size_t)k0, kc, n0D, tr);
          });
        s->step_counter = save;
        if (!rc && hipEventRecord(s->adj_ev[2 + buf], s->stream) != hipSuccess) rc = FMS_ERR_HIP;
        s->stream = main_stream;
        if (rc) break;
        // reverse the segment on the solver's stream once its tape is recorded
        if (hipStreamWaitEvent(s->stream, s->adj_ev[2 + buf], 0) != hipSuccess) {
          rc = fail(FMS_ERR_HIP, "hipStreamWaitEvent failed");
          break;
        }
      }
      fms::AdjArgs args{};
      args.fb = s->fibers();
      args.st = fms::AdjStim{s->stim_mode == FMS_STIM_CURRENT, s->stim_param, s->d_onset, s->d_dur, s->d_amp,
                             s->vc_width > 0 ? s->d_vc_centre : nullptr};
      args.tape = tape;
      args.steps = s->d_steps + 4 * (size_t)k0;
      args.kc = kc;
      args.n0D = n0D;
      args.ie = ie;
      args.sensor_slot = s->d_sensor_slot;
      args.dtrace = d_dtraces + (size_t)k0 * F * S;
      args.n_sensors = S;
      args.lam = s->d_lam;
      args.acc = s->d_gacc;
      args.raise_priority = !whole && s->tune_adjoint == FMS_ADJOINT_OVERLAP_PRIORITY;
      fms::adjoint_launch<E>(T, s->nmax, args, s->stream);
      if (hipGetLastError() != hipSuccess) {
        rc = fail(FMS_ERR_HIP, "adjoint kernel launch failed");
        break;
      }
      if (!whole && hipEventRecord(s->adj_ev[buf], s->stream) != hipSuccess) {
        rc = fail(FMS_ERR_HIP, "hipEventRecord failed");
        break;
      }
    }
    s->stream = main_stream;
    if (rc && !whole) (void)hipStreamSynchronize(s->stream2);
    s->spikes = saved_spikes;
    s->tune_resident = saved_resident;
    if (rc) return rc;
    hipLaunchKernelGGL(fms::k_adj_reduce, dim3(F), dim3(256), 0, s->stream, F, T, s->d_gacc, ie ? 1.0 : 0.5, s->d_grad,
                       s->d_pfbar);
    HIP_TRY(hipGetLastError());
    return 0;
  }
}

int adjoint_backward(FmsSolver *s, const double *d_dtraces) {
  return s->exp_mode == FMS_EXP_APPROXIMATE ? adjoint_backward_core<fms::ExpApproxFma>(s, d_dtraces)
                                            : adjoint_backward_core<fms::ExpLibmFma>(s, d_dtraces);
}

// forward over all segments, checkpointing; traces go to device memory d_traces
int adjoint_forward(FmsSolver *s, const double *steps, int n_steps, int n0D, int checkpoint_interval,
                    double *d_traces) {
  if (!s || !steps || n_steps <= 0 || n0D < 1 || checkpoint_interval < 1)
    return fail(FMS_ERR_ARGUMENT, "bad adjoint forward arguments");
  if (s->n_sensors <= 0) return fail(FMS_ERR_STATE, "call fms_set_sensors first");
  if (s->precision != FMS_FP64) return fail(FMS_ERR_UNSUPPORTED, "the adjoint runs in FP64");
  if (s->stim_mode == FMS_STIM_FIRING_TABLE)
    return fail(FMS_ERR_UNSUPPORTED, "the Vm clamp of firing-table stimulation is not differentiable; use current pulses");
  if (s->only_if_stimulated) return fail(FMS_ERR_UNSUPPORTED, "onlyComputeIfHasBeenStimulated is not differentiable");
  if (s->nmax > 2048) return fail(FMS_ERR_UNSUPPORTED, "the adjoint takes fibres of <= 2048 nodes");
  const int F = s->F, S = s->n_sensors, K = n_steps, Kc = checkpoint_interval;
  const int nseg = (K + Kc - 1) / Kc;
  int rc;
  // the whole tape (step k's entries at k * (2 NS + 1) * N, the layout the
  // backward's recompute writes into a segment buffer), or a checkpoint per
  // segment of Kc steps
  const long long step_len = (long long)(2 * Model::NS + 1) * s->N;
  const long long whole_len = (long long)K * step_len;
  bool whole = s->tune_adjoint_tape == FMS_ADJOINT_TAPE_WHOLE;
  if (s->tune_adjoint_tape == FMS_ADJOINT_TAPE_AUTO) {
    size_t free_b = 0, total_b = 0;
    HIP_TRY(hipMemGetInfo(&free_b, &total_b));
    // the tape held now is freed before a larger one is allocated
    const double avail = (double)free_b + (double)s->tape_cap * sizeof(double);
    whole = (double)whole_len * sizeof(double) <= 0.5 * avail;
  }
  s->adj_whole = 0;
  s->adj_K = 0;   // no backward until this forward has been enqueued
  if (whole && (rc = ensure(&s->d_tape, s->tape_cap, whole_len))) return rc;
  if (!whole && (rc = ensure(&s->d_ckpt, s->ckpt_cap, (long long)(nseg * ckpt_doubles(s))))) return rc;
  // a whole tape of an earlier forward is released when checkpoints take over
  // (the backward then needs two segment buffers only)
  if (!whole && s->tape_cap > 2 * (long long)Kc * step_len) {
    HIP_TRY(hipFree(s->d_tape));
    s->d_tape = nullptr;
    s->tape_cap = 0;
  }
  if ((rc = upload_steps(s, steps, K, false))) return rc;
  s->adj_steps.assign(steps, steps + 4 * (size_t)K);
  s->adj_n0D = n0D;
  s->adj_interval = Kc;
  // with the whole tape nothing ties a launch to a segment: the solver's
  // steps per fused launch
  const int len = whole ? fibre_launch_steps(s, std::min(s->tune_chunk, K), n0D, FIBRE_FLAG_BYTES) : Kc;
  if (ensure_flag_bytes(s, fibre_flag_bytes(s, std::min(len, K), n0D))) return FMS_ERR_HIP;
  for (int seg = 0; seg * (long long)len < K; seg++) {
    const int k0 = seg * len, kc = std::min(len, K - k0);
    if (!whole && (rc = copy_state(s, s->d_ckpt + (size_t)seg * ckpt_doubles(s), true))) return rc;
    fms::DevTrace tr{};
    if (whole) tr.tape = s->d_tape + (size_t)k0 * (size_t)step_len;
    tr.sensor_slot = s->d_sensor_slot;
    tr.trace = d_traces + (size_t)k0 * F * S;
    tr.n_sensors = S;
    rc = with_exp(s, [&](auto e) {
      return launch_fused<double, decltype(e)>(s, s->d_steps + 4 * (size_t)k0, kc, n0D, tr);
    });
    if (rc) return rc;
  }
  s->adj_whole = whole;
  s->adj_K = K;
  return 0;
}

}  // namespace

extern "C" {

int fms_set_parameters(FmsSolver *s, const double *params, const double *prefactor) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (params && Model::NP > 0)
    HIP_TRY(hipMemcpy(s->d_params, params, (size_t)s->F * Model::NP * sizeof(double), hipMemcpyHostToDevice));
  if (prefactor) HIP_TRY(hipMemcpy(s->d_pf, prefactor, (size_t)s->F * sizeof(double), hipMemcpyHostToDevice));
  return 0;
  FMS_API_END
}

int fms_set_sensors(FmsSolver *s, const int *sensor_nodes, int n_sensors) {
  FMS_API_BEGIN
  if (!s || n_sensors < 0 || (n_sensors > 0 && !sensor_nodes)) return fail(FMS_ERR_ARGUMENT, "bad sensors");
  const int F = s->F;
  std::vector<int> slot((size_t)s->N, -1);
  for (int f = 0; f < F; f++) {
    const int n = s->h_off[f + 1] - s->h_off[f];
    for (int j = 0; j < n_sensors; j++) {
      const int i = sensor_nodes[(size_t)f * n_sensors + j];
      if (i < 0 || i >= n) return fail(FMS_ERR_ARGUMENT, "sensor node outside its fibre");
      if (slot[(size_t)s->h_off[f] + i] >= 0) return fail(FMS_ERR_ARGUMENT, "duplicate sensor node");
      slot[(size_t)s->h_off[f] + i] = j;
    }
  }
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (s->d_sensor_nodes) HIP_TRY(hipFree(s->d_sensor_nodes));
  if (s->d_sensor_slot) HIP_TRY(hipFree(s->d_sensor_slot));
  s->d_sensor_nodes = nullptr;
  s->d_sensor_slot = nullptr;
  s->n_sensors = n_sensors;
  if (n_sensors == 0) return 0;
  if (dalloc(&s->d_sensor_nodes, (size_t)F * n_sensors) || dalloc(&s->d_sensor_slot, (size_t)s->N)) return FMS_ERR_HIP;
  HIP_TRY(hipMemcpy(s->d_sensor_nodes, sensor_nodes, (size_t)F * n_sensors * sizeof(int), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(s->d_sensor_slot, slot.data(), (size_t)s->N * sizeof(int), hipMemcpyHostToDevice));
  return 0;
  FMS_API_END
}

int fms_adjoint_forward(FmsSolver *s, const double *steps, int n_steps, int n0D, int checkpoint_interval,
                        double *traces) {
  FMS_API_BEGIN
  if (!s) return fail(FMS_ERR_ARGUMENT, "null solver");
  int rc;
  if (n_steps > 0 && s->n_sensors > 0 &&
      (rc = ensure(&s->d_trace, s->trace_cap, (long long)n_steps * s->F * s->n_sensors)))
    return rc;
  if ((rc = adjoint_forward(s, steps, n_steps, n0D, checkpoint_interval, s->d_trace))) return rc;
  if (traces) {
    HIP_TRY(hipStreamSynchronize(s->stream));
    HIP_TRY(hipMemcpy(traces, s->d_trace, (size_t)n_steps * s->F * s->n_sensors * sizeof(double),
                      hipMemcpyDeviceToHost));
  }
  return 0;
  FMS_API_END
}

int fms_adjoint_forward_device(FmsSolver *s, const double *steps, int n_steps, int n0D, int checkpoint_interval,
                               double *d_traces) {
  FMS_API_BEGIN
  if (!s || !d_traces) return fail(FMS_ERR_ARGUMENT, "null argument");
  int rc;
  if ((rc = adjoint_forward(s, steps, n_steps, n0D, checkpoint_interval, d_traces))) return rc;
  HIP_TRY(hipStreamSynchronize(s->stream));
  return 0;
  FMS_API_END
}

int fms_adjoint_backward(FmsSolver *s, const double *dtraces, double *grad_params, double *grad_prefactor) {
  FMS_API_BEGIN
  if (!s || !dtraces) return fail(FMS_ERR_ARGUMENT, "null argument");
  if (s->adj_K <= 0) return fail(FMS_ERR_STATE, "call fms_adjoint_forward first");
  const size_t len = (size_t)s->adj_K * s->F * s->n_sensors;
  long long cap = 0;
  int rc;
  if ((rc = ensure(&s->d_dtrace, cap, (long long)len))) return rc;
  HIP_TRY(hipMemcpyAsync(s->d_dtrace, dtraces, len * sizeof(double), hipMemcpyHostToDevice, s->stream));
  if ((rc = adjoint_backward(s, s->d_dtrace))) return rc;
  HIP_TRY(hipStreamSynchronize(s->stream));
  if (grad_params) HIP_TRY(hipMemcpy(grad_params, s->d_grad, 3 * (size_t)s->F * sizeof(double), hipMemcpyDeviceToHost));
  if (grad_prefactor)
    HIP_TRY(hipMemcpy(grad_prefactor, s->d_pfbar, (size_t)s->F * sizeof(double), hipMemcpyDeviceToHost));
  return 0;
  FMS_API_END
}

int fms_adjoint_whole_tape(FmsSolver *s, int *whole) {
  FMS_API_BEGIN
  if (!s || !whole) return fail(FMS_ERR_ARGUMENT, "null argument");
  if (s->adj_K <= 0) return fail(FMS_ERR_STATE, "call fms_adjoint_forward first");
  *whole = s->adj_whole;
  return 0;
  FMS_API_END
}

int fms_adjoint_backward_device(FmsSolver *s, const double *d_dtraces, double *d_grad_params,
                                double *d_grad_prefactor) {
  FMS_API_BEGIN
  if (!s || !d_dtraces) return fail(FMS_ERR_ARGUMENT, "null argument");
  if (s->adj_K <= 0) return fail(FMS_ERR_STATE, "call fms_adjoint_forward first");
  int rc;
  if ((rc = adjoint_backward(s, d_dtraces))) return rc;
  if (d_grad_params)
    HIP_TRY(hipMemcpyAsync(d_grad_params, s->d_grad, 3 * (size_t)s->F * sizeof(double), hipMemcpyDeviceToDevice,
                           s->stream));
  if (d_grad_prefactor)
    HIP_TRY(hipMemcpyAsync(d_grad_prefactor, s->d_pfbar, (size_t)s->F * sizeof(double), hipMemcpyDeviceToDevice,
                           s->stream));
  HIP_TRY(hipStreamSynchronize(s->stream));
  return 0;
  FMS_API_END
}

}  // extern "C"

// ===========================================================================
// autotuner: times the schedules that give bit-identical results on the
// solver's own batch and keeps the fastest
// ===========================================================================
namespace {

// device state that a trial run changes: states, the stimulation state
// machine, the stimulation log counter and the spike detector
struct Snapshot {
  std::vector<std::pair<void *, size_t>> regions;
  std::vector<void *> copies;
  long long step_counter = 0, n_fused = 0, n_reaction = 0, n_thomas = 0, n_gcap = 0, n_glaunch = 0;
};

int snapshot_take(FmsSolver *s, Snapshot &sn) {
  const size_t N = (size_t)s->N, F = (size_t)s->F;
  auto add = [&](void *p, size_t bytes) {
    if (p && bytes) sn.regions.push_back({p, bytes});
  };
  add(s->d_vm, N * sizeof(double));
  add(s->d_gates, (size_t)(Model::NS - 1) * s->GS * gate_bytes(s));
  add(s->d_last, F * sizeof(double));
  add(s->d_curjit, F * sizeof(double));
  add(s->d_jidx, F * sizeof(int));
  add(s->d_curr, F);
  add(s->d_hasbeen, F);
  add(s->d_log_count, sizeof(int));
  if (s->spikes) {
    add(s->d_vprev, N * sizeof(double));
    add(s->d_sfirst, N * sizeof(int));
    add(s->d_scount, N * sizeof(int));
  }
  for (auto &r : sn.regions) {
    void *c = nullptr;
    HIP_TRY(hipMalloc(&c, r.second));
    sn.copies.push_back(c);
    HIP_TRY(hipMemcpyAsync(c, r.first, r.second, hipMemcpyDeviceToDevice, s->stream));
  }
  sn.step_counter = s->step_counter;
  sn.n_fused = s->n_launch_fused;
  sn.n_reaction = s->n_launch_reaction;
  sn.n_thomas = s->n_launch_thomas;
  sn.n_gcap = s->n_graph_captures;
  sn.n_glaunch = s->n_graph_launches;
  return 0;
}

int snapshot_restore(FmsSolver *s, const Snapshot &sn) {
  for (size_t k = 0; k < sn.regions.size(); k++)
    HIP_TRY(hipMemcpyAsync(sn.regions[k].first, sn.copies[k], sn.regions[k].second, hipMemcpyDeviceToDevice,
                           s->stream));
  s->step_counter = sn.step_counter;
  s->n_launch_fused = sn.n_fused;
  s->n_launch_reaction = sn.n_reaction;
  s->n_launch_thomas = sn.n_thomas;
  s->n_graph_captures = sn.n_gcap;
  s->n_graph_launches = sn.n_glaunch;
  return 0;
}

void snapshot_free(Snapshot &sn) {
  for (void *c : sn.copies)
    if (c) (void)hipFree(c);
  sn.copies.clear();
}

// Digest of the device state a trial leaves behind, to check that a candidate
// schedule computed the same bits as the solver's own schedule. Each region's
// 8-byte words are mixed with their position and summed (mod 2^64), so the
// reduction order does not matter; the stimulation log, whose entries land in
// atomic order, enters as an order-free sum over its (time, fibre) pairs.
__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
  z += 0x9e3779b97f4a7c15ULL;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}

__device__ __forceinline__ void digest_add(unsigned long long acc, unsigned long long *out) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if ((threadIdx.x & 63) == 0) atomicAdd(out, acc);
}

__global__ void k_digest(const unsigned char *p, unsigned long long bytes, unsigned long long salt,
                         unsigned long long *out) {
  const unsigned long long nw = bytes / 8;
  const unsigned long long *w = reinterpret_cast<const unsigned long long *>(p);
  unsigned long long acc = 0;
  for (unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; i < nw;
       i += (unsigned long long)gridDim.x * blockDim.x)
    acc += mix64(w[i] ^ mix64(i + salt));
  if (blockIdx.x == 0 && threadIdx.x == 0 && bytes % 8) {
    unsigned long long t = 0;
    for (unsigned long long k = nw * 8; k < bytes; k++) t = (t << 8) | p[k];
    acc += mix64(t ^ mix64(nw + salt));
  }
  digest_add(acc, out);
}

__global__ void k_digest_log(const double *times, const int *fibers, const int *count, int cap,
                             unsigned long long *out) {
  const int n = min(*count, cap);
  unsigned long long acc = 0;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x)
    acc += mix64((unsigned long long)__double_as_longlong(times[k]) ^ mix64((unsigned long long)(unsigned)fibers[k]));
  digest_add(acc, out);
}

int state_digest(FmsSolver *s, const Snapshot &sn, unsigned long long *d_out, unsigned long long &h) {
  HIP_TRY(hipMemsetAsync(d_out, 0, sizeof(unsigned long long), s->stream));
  for (size_t k = 0; k < sn.regions.size(); k++) {
    const unsigned long long bytes = sn.regions[k].second;
    const unsigned blocks = (unsigned)std::min<unsigned long long>(1024, (bytes / 8 + 255) / 256 + 1);
    hipLaunchKernelGGL(k_digest, dim3(blocks), dim3(256), 0, s->stream, (const unsigned char *)sn.regions[k].first,
                       bytes, (unsigned long long)(k + 1) << 40, d_out);
    HIP_TRY(hipGetLastError());
  }
  if (s->stim_mode == FMS_STIM_FIRING_TABLE && s->log_cap > 0 && s->d_log_count) {
    hipLaunchKernelGGL(k_digest_log, dim3(64), dim3(256), 0, s->stream, s->d_log_time, s->d_log_fiber,
                       s->d_log_count, s->log_cap, d_out);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipMemcpyAsync(&h, d_out, sizeof(h), hipMemcpyDeviceToHost, s->stream));
  HIP_TRY(hipStreamSynchronize(s->stream));
  return 0;
}

struct Schedule {
  int kernels, chunk, resident, threads, graph, per_fibre, rthreads;
};

int apply_schedule(FmsSolver *s, const Schedule &c) {
  s->kernels = c.kernels;
  s->tune_chunk = c.chunk;
  s->tune_resident = c.resident;
  s->tune_threads = c.threads;
  s->tune_graph = c.graph;
  s->tune_reaction_fibre = c.per_fibre;
  s->tune_reaction_threads = c.rthreads;
  if (c.kernels == FMS_KERNELS_SPLIT && s->thomas == FMS_THOMAS_SERIAL && !s->d_cA) {
    if (dalloc(&s->d_cA, (size_t)s->N) || dalloc(&s->d_dA, (size_t)s->N)) return FMS_ERR_HIP;
  }
  return 0;
}

// candidates in the order they are tried; every one computes the same
// arithmetic in the same order (bit-identical states)
std::vector<Schedule> candidates(const FmsSolver *s, int allow_split) {
  std::vector<Schedule> v;
  const bool small = Model::NS <= 8 && s->nmax <= 2048;
  const bool fused_ok = !(s->nmax > 2048 && s->thomas == FMS_THOMAS_SERIAL) && s->nmax <= 4096;
  const int pf = s->tune_reaction_fibre, rt = s->tune_reaction_threads;
  if (fused_ok) {
    if (small && s->thomas == FMS_THOMAS_PARTITIONED) {
      // the gates stay in registers: only the launches' length is left
      for (int chunk : {64, 256, 512}) v.push_back({FMS_KERNELS_FUSED, chunk, 1, 256, 0, pf, rt});
    } else if (small) {
      for (int chunk : {64, 512}) {
        v.push_back({FMS_KERNELS_FUSED, chunk, 1, 256, 0, pf, rt});
        v.push_back({FMS_KERNELS_FUSED, chunk, 0, 256, 0, pf, rt});
        // the partitioned solve's elimination order depends on the threads per
        // fibre, so 128-thread schedules are bit-identical only with the serial solve
        if (s->nmax <= 1024) {
          v.push_back({FMS_KERNELS_FUSED, chunk, 1, 128, 0, pf, rt});
          v.push_back({FMS_KERNELS_FUSED, chunk, 0, 128, 0, pf, rt});
        }
      }
    } else {
      v.push_back({FMS_KERNELS_FUSED, 512, 0, 256, 0, pf, rt});
    }
  }
  if (allow_split || !fused_ok) {
    if (Model::NS > 8) {
      // reaction per fibre (workgroups of 256 or 64 threads) or per node
      for (int r : {256, 64})
        for (int g : {0, 8}) v.push_back({FMS_KERNELS_SPLIT, s->tune_chunk, s->tune_resident, 256, g, 1, r});
      for (int g : {0, 8}) v.push_back({FMS_KERNELS_SPLIT, s->tune_chunk, s->tune_resident, 256, g, 0, rt});
    } else {
      for (int g : {0, 8, 32}) v.push_back({FMS_KERNELS_SPLIT, s->tune_chunk, s->tune_resident, 256, g, pf, rt});
    }
  }
  return v;
}

}  // namespace

extern "C" {

int fms_autotune(FmsSolver *s, const double *steps, int n_steps, int n0D, int allow_split, FmsTuneResult *result,
                 double *candidate_ms, int capacity) {
  FMS_API_BEGIN
  if (!s || !steps || n_steps < 1 || n0D < 1) return fail(FMS_ERR_ARGUMENT, "bad autotune arguments");
  if (s->d_alg) return fail(FMS_ERR_STATE, "autotune before requesting algebraics for transfer");
  const std::vector<Schedule> cand = candidates(s, allow_split);
  if (cand.empty()) return fail(FMS_ERR_UNSUPPORTED, "no schedule fits this batch");
  const Schedule keep{s->kernels, s->tune_chunk, s->tune_resident, s->tune_threads, s->tune_graph,
                      s->tune_reaction_fibre, s->tune_reaction_threads};
  Snapshot sn;
  int rc = snapshot_take(s, sn);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (!rc && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess))
    rc = fail(FMS_ERR_HIP, "hipEventCreate failed");
  int best = -1, rejected = 0;
  double best_ms = 0;
  // the solver's own schedule computes the reference digest
  unsigned long long *d_digest = nullptr, ref_digest = 0;
  if (!rc) rc = dalloc(&d_digest, 1);
  if (!rc) rc = snapshot_restore(s, sn);
  if (!rc) rc = dispatch(s, steps, n_steps, n0D);
  if (!rc) rc = state_digest(s, sn, d_digest, ref_digest);
  for (size_t k = 0; k < cand.size() && !rc; k++) {
    if ((rc = apply_schedule(s, cand[k]))) break;
    // one untimed pass (graph capture, code object load), then the timed pass
    for (int pass = 0; pass < 2 && !rc; pass++) {
      if ((rc = snapshot_restore(s, sn))) break;
      if (pass == 1 && hipEventRecord(e0, s->stream) != hipSuccess) rc = fail(FMS_ERR_HIP, "hipEventRecord");
      if (!rc) rc = dispatch(s, steps, n_steps, n0D);
      if (!rc && pass == 1 && hipEventRecord(e1, s->stream) != hipSuccess) rc = fail(FMS_ERR_HIP, "hipEventRecord");
    }
    if (rc) break;
    if (hipEventSynchronize(e1) != hipSuccess) {
      rc = fail(FMS_ERR_HIP, "hipEventSynchronize");
      break;
    }
    float ms = 0;
    (void)hipEventElapsedTime(&ms, e0, e1);
    // a candidate whose states, stimulation state machine, log or spike data
    // differ from the solver's own schedule's is reported (negative time) and
    // never chosen
    unsigned long long dig = 0;
    if ((rc = state_digest(s, sn, d_digest, dig))) break;
    const bool same = dig == ref_digest;
    if (candidate_ms && (int)k < capacity) candidate_ms[k] = same ? ms / n_steps : -1.0;
    if (!same) {
      rejected++;
      continue;
    }
    if (best < 0 || ms < best_ms) {
      best = (int)k;
      best_ms = ms;
    }
  }
  if (d_digest) (void)hipFree(d_digest);
  if (!rc) rc = snapshot_restore(s, sn);
  if (!rc && hipStreamSynchronize(s->stream) != hipSuccess) rc = fail(FMS_ERR_HIP, "hipStreamSynchronize");
  snapshot_free(sn);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (rc) {
    (void)apply_schedule(s, keep);
    return rc;
  }
  // every candidate rejected: the solver keeps its own schedule
  const Schedule chosen = best >= 0 ? cand[best] : keep;
  if ((rc = apply_schedule(s, chosen))) return rc;
  if (result) {
    result->kernels = chosen.kernels;
    result->steps_per_launch = chosen.chunk;
    result->resident_gates = chosen.resident;
    result->threads = chosen.threads;
    result->graph_steps = chosen.graph;
    result->reaction_per_fibre = chosen.per_fibre;
    result->reaction_threads = chosen.rthreads;
    result->ms_per_step = best >= 0 ? best_ms / n_steps : -1.0;
    result->n_candidates = (int)cand.size();
    result->n_rejected = rejected;
  }
  return 0;
  FMS_API_END
}

}  // extern "C"
