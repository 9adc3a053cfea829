// Resident fused kernel of the small models (at most 8 states, partitioned
// solve): one workgroup per fibre runs many split steps and reads and writes the
// fibre's state once.
//
//  * Thread t owns the c = ceil(n / T) consecutive nodes from t*c on, for the
//    reaction and for the diffusion (fms_chunk.h) alike: Vm and gates stay with it
//    between two launches, and the diffusion's coefficients beside them as long as dt
//    does not change. One barrier per split step. The kernel is compiled for two waves
//    per SIMD, 256 registers; with 5 to 8 nodes per thread about 40 values are spilled
//    to scratch.
//  * Waves past the fibre's end skip the reaction; threads past it shadow its
//    last node and store nothing.
//  * Nodes are advanced one after the other (two per basic block gained nothing at two
//    waves per SIMD); a stimulus's selects stand behind a branch that only the waves
//    with stimulated nodes take, while the stimulus is on.
//  * The stimulation state machine does not depend on the states: k_fibre_flags
//    evaluates it for the whole launch beforehand, one wave per fibre, 64 Heun
//    steps at a time.
//
// Bound by FP64 instruction issue: the two reaction halves are about 450
// instructions per node and step, the solve about 15.
#pragma once

#include "fms_chunk.h"
#include "fms_fused.h"

namespace fms {

// flags of 64 consecutive Heun steps of one fibre (per split step the n0D of the
// first half, then the n0D of the second): bit i of `stim` says whether the
// stimulus is on, of `compute` whether the reaction runs
struct FlagGroup {
  unsigned long long stim, compute;
};

__host__ __device__ constexpr long long flag_groups(long long steps, int n0D) { return (steps * 2 * n0D + 63) / 64; }

// The state machine of stim_flag for the K split steps from `steps` on, one wave
// per fibre. Lane i evaluates Heun step i of each group of 64 against the state
// machine's current state; at the first lane whose check changes that state
// (repeat time over: next period, next jitter value) the lanes before it are
// final, the state advances and the lanes after it are evaluated again: the same
// checks on the same values as one thread going through the steps in time order,
// whose chain of global loads per step the fused kernel had waited for.
static __global__ __launch_bounds__(64) void k_fibre_flags(DevStim st, const double *__restrict__ steps, int K, int n0D,
                                                    FlagGroup *__restrict__ flags) {
  const int f = blockIdx.x, lane = threadIdx.x;
  const long long count = (long long)K * 2 * n0D, groups = flag_groups(K, n0D);
  FlagGroup *out = flags + f * groups;
  const bool only = st.only_if_stimulated != 0;
  bool hb = st.has_been[f] != 0;
  const bool hb_start = hb;
  const bool checked = stim_checked(st, f), table = checked && st.mode == 1;
  double freq = 0, repeat = 0, begin = 0, last = 0, jit = 0;
  int col = 0, jidx = 0, currently = 0;
  if (table) {
    freq = st.freq[f];
    repeat = st.repeat[f];
    begin = st.enable_begin[f];
    col = st.motor_unit[f] % st.fe_cols;
    last = st.last_check[f];
    jit = st.cur_jitter[f];
    jidx = st.jitter_idx[f];
    currently = st.currently[f];
  }
  for (long long gi = 0; gi < groups; gi++) {
    const long long i = gi * 64 + lane;
    const bool active = i < count;
    double t = 0.0;
    if (active) {
      const long long s = i / (2 * n0D);
      const int r = (int)(i - s * 2 * n0D);
      const double *row = steps + 4 * s;
      t = half_start(row, r / n0D) + (r % n0D) * row[2];
    }
    int stim = 0;
    if (table) {
      int fires = 0;
      if (active) {
        const int idx = (int)round(t * freq);
        const unsigned long fr = (unsigned long)(long)idx % (unsigned long)st.fe_rows;
        fires = st.firing_events[fr * st.fe_cols + col];
      }
      int done = 0;   // lanes before it are final
      while (done < 64) {
        const double next = last + 1. / (freq + jit);
        const bool due = active && lane >= done && t >= next && t >= begin - 1e-13;
        const bool change = due && repeat != 0 && t - next > repeat;
        const unsigned long long mc = __builtin_amdgcn_ballot_w64(change);
        const int first = mc ? __builtin_ctzll(mc) : 64;
        if (lane >= done && lane < first) stim = due && fires;
        if (first < 64) {
          last += 1. / (freq + jit);
          double jf = 0.0;
          if (st.jitter_cnt[f] > 0) jf = st.jitter[st.jitter_off[f] + jidx % st.jitter_cnt[f]];
          jit = jf * freq;
          jidx++;
        }
        done = first + 1;
      }
    } else if (checked && st.mode == 2) {
      stim = active && current_on(st, f, t);
    }
    const unsigned long long m = __builtin_amdgcn_ballot_w64(stim != 0);
    if (table) {
      // rising edges: stimulated now and not at the step before
      const unsigned long long rise = m & ~((m << 1) | (currently ? 1ULL : 0ULL));
      if (rise && st.log_count) {
        int k0 = 0;
        if (lane == 0) k0 = atomicAdd(st.log_count, __builtin_popcountll(rise));
        k0 = __shfl(k0, 0);
        const int k = k0 + __builtin_popcountll(rise & ((1ULL << lane) - 1));
        if (((rise >> lane) & 1) && k < st.log_cap) {
          st.log_time[k] = t;
          st.log_fiber[k] = f;
        }
      }
      const int last_lane = count - gi * 64 < 64 ? (int)(count - gi * 64) - 1 : 63;
      currently = (int)((m >> last_lane) & 1);
    }
    // the fibre computes from the Heun step of its first stimulation on
    const unsigned long long since = m ? ~0ULL << __builtin_ctzll(m) : 0ULL;
    if (lane == 0) out[gi] = FlagGroup{m, !only || hb ? ~0ULL : since};
    hb = hb || m != 0;
  }
  if (lane == 0) {
    if (table) {
      st.last_check[f] = last;
      st.cur_jitter[f] = jit;
      st.jitter_idx[f] = jidx;
      st.currently[f] = (unsigned char)currently;
    }
    if (hb && !hb_start) st.has_been[f] = 1;
  }
}

// what the fused kernel needs of the stimulation
struct FibreStim {
  int clamp;        // the stimulus sets Vm to vstim (firing table), else parameter `param` to the amplitude
  int param;
  double vstim;
  const double *amplitude;   // [F], current pulses
  const FlagGroup *flags;    // [F][flag_groups(K, n0D)]
};

// One Heun step of the thread's nodes. `on`: the stimulus is on and the wave holds
// stimulated nodes (bits of `inset`); it is uniform over the wave, so the selects it
// needs cost the other steps a branch.
template <class M, class G, class E, int C>
__device__ __forceinline__ void fibre_heun(double *V, G (*g)[M::NS - 1], const double *p, double t, double dt, bool on,
                                           unsigned inset, const FibreStim &st, double amplitude) {
  if constexpr (std::is_same<M, ModelHH>::value) {
    if (!on || st.clamp || st.param == 0) {
      constexpr_for<0, C, 1>([&](auto k_) {
        constexpr int k = decltype(k_)::value;
        double i_stim = p[0];
        if (on && !st.clamp) i_stim = (inset >> k) & 1 ? amplitude : p[0];
        hh_step<G, E, false>(V[k], g[k], p, i_stim, dt,
                             [&](double &v) {
                               if (on && st.clamp) v = (inset >> k) & 1 ? st.vstim : v;
                             },
                             nullptr);
        if (on && st.clamp) V[k] = (inset >> k) & 1 ? st.vstim : V[k];
      });
      return;
    }
  }
  // other models, and a stimulus on another parameter
  constexpr_for<0, C, 1>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    const bool in = on && ((inset >> k) & 1);
    double pk[M::NP > 0 ? M::NP : 1];
#pragma unroll
    for (int q = 0; q < M::NP; q++) pk[q] = in && !st.clamp && q == st.param ? amplitude : p[q];
    heun_node<M, G, E, false>(V[k], g[k], pk, t, dt, in && st.clamp, st.vstim);
  });
}

// C consecutive doubles of a thread's nodes to the tape, two per store (8-byte
// aligned: one store per node left each cache line to C partial writes)
typedef double double2_a8 __attribute__((ext_vector_type(2), aligned(8)));
template <int C> __device__ __forceinline__ void tape_row(double *dst, int lo, int n, const double *v) {
  constexpr_for<0, C, 2>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    if constexpr (k + 1 < C) {
      if (lo + k + 1 < n) {
        *reinterpret_cast<double2_a8 *>(dst + k) = double2_a8{v[k], v[k + 1]};
        return;
      }
    }
    if (lo + k < n) dst[k] = v[k];
  });
}
// Vm and the gates
template <class M, class G, int C>
__device__ __forceinline__ void tape_state(double *dst, long long N, int lo, int n, const double *V,
                                           const G (*g)[M::NS - 1]) {
  tape_row<C>(dst, lo, n, V);
#pragma unroll
  for (int q = 0; q < M::NS - 1; q++) {
    double v[C];
#pragma unroll
    for (int k = 0; k < C; k++) v[k] = (double)g[k][q];
    tape_row<C>(dst + (q + 1) * N, lo, n, v);
  }
}

// the fibre's steps with C nodes per thread; TAPE: sensor traces and the adjoint's
// tape are recorded (either may be absent)
template <class M, class G, class E, int T, int C, bool TAPE>
__device__ __forceinline__ void fibre_steps(const DevFibers &fb, const FibreStim &st, double *__restrict__ vm,
                                            G *__restrict__ gates, const double *__restrict__ steps, int K, int n0D,
                                            int ie, const DevSpikes &spk, const DevTrace &tr, int f, int off, int n,
                                            double *sh) {
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double pf = fb.prefactor[f];
  const ChunkLds<T, C> lds{sh, tid};
  const int lo = tid * C;
  const bool busy = wave * 64 * C < n;   // the wave holds nodes of the fibre
  const FlagGroup *flags = st.flags + f * flag_groups(K, n0D);

  double p[M::NP > 0 ? M::NP : 1];
#pragma unroll
  for (int k = 0; k < M::NP; k++) p[k] = fb.params[(long long)f * M::NP + k];
  double V[C];
  G g[C][M::NS - 1];
  unsigned inset = 0, below = 0, sensor = 0;
  {
    const int sb = fb.stim_begin[f], se = fb.stim_end[f];
#pragma unroll
    for (int k = 0; k < C; k++) {
      const int i = off + (lo + k < n ? lo + k : n - 1);
      V[k] = vm[i];
#pragma unroll
      for (int q = 0; q < M::NS - 1; q++) g[k][q] = gates[(long long)q * fb.gate_stride + i];
      if (lo + k < n) {
        inset |= (lo + k >= sb && lo + k < se ? 1u : 0u) << k;
        // bit k of `below`: node k was below the threshold at the last check
        if (spk.enabled) below |= (spk.vm_prev[i] < spk.threshold ? 1u : 0u) << k;
        if (TAPE && tr.sensor_slot) sensor |= (tr.sensor_slot[i] >= 0 ? 1u : 0u) << k;
      }
    }
  }
  const bool wave_inset = __builtin_amdgcn_ballot_w64(inset != 0) != 0;

  // the thread's first node in row `slot` of step s's tape
  auto tape_at = [&](int s, int slot) {
    return tr.tape + ((long long)s * (2 * M::NS + 1) + slot) * fb.n_total + off + lo;
  };
  // half step hs: the first reaction half of step hs / 2, or (odd) its diffusion
  // and second reaction half. The outer loop runs once per change of dt.
  int hs = 0;
  FlagGroup fl{0, 0};
  while (hs < 2 * K) {
    const double dt1 = steps[4 * (long long)(hs >> 1) + 3];
    ChunkFactor<C> fac;
    chunk_refactor<T, C>(fac, n, fb.elem_len + (off - f), pf, dt1, ie != 0, lds);
#pragma unroll 1
    do {
      const int s = hs >> 1;
      const bool half = hs & 1;
      const double *row = steps + 4 * (long long)s;
      if (half) chunk_diffuse<T, C>(fac, V, s & 1, lds);
      if (TAPE && tr.tape) {
        // half 0: the state before it; half 1: Vm after the diffusion
        if (half)
          tape_row<C>(tape_at(s, 2 * M::NS), lo, n, V);
        else
          tape_state<M, G, C>(tape_at(s, 0), fb.n_total, lo, n, V, g);
      }
      if (busy) {
        const double t0 = half_start(row, half), dt = row[2];
#pragma unroll 1
        for (int j = 0; j < n0D; j++) {
          const int q = hs * n0D + j;
          if ((q & 63) == 0) fl = flags[q >> 6];
          if (!((fl.compute >> (q & 63)) & 1)) continue;
          const bool on = wave_inset && ((fl.stim >> (q & 63)) & 1);
          fibre_heun<M, G, E, C>(V, g, p, t0 + j * dt, dt, on, inset, st, on && !st.clamp ? st.amplitude[f] : 0.0);
        }
      }
      if (TAPE && tr.tape && !half) tape_state<M, G, C>(tape_at(s, M::NS), fb.n_total, lo, n, V, g);
      if (half && TAPE && sensor) {
#pragma unroll
        for (int k = 0; k < C; k++)
          if ((sensor >> k) & 1)
            tr.trace[((long long)s * fb.n_fibers + f) * tr.n_sensors + tr.sensor_slot[off + lo + k]] = V[k];
      }
      if (half && spk.enabled && busy) {
        unsigned now = 0;
#pragma unroll
        for (int k = 0; k < C; k++) now |= (V[k] < spk.threshold ? 1u : 0u) << k;
        // nodes that were below the threshold and are not (a NaN is no crossing)
        const unsigned cross = below & ~now;
        below = now;
        if (cross) {
#pragma unroll
          for (int k = 0; k < C; k++)
            if (((cross >> k) & 1) && lo + k < n && V[k] >= spk.threshold) {
              const int i = off + lo + k;
              spk.count[i]++;
              if (spk.first_step[i] < 0) spk.first_step[i] = spk.step0 + s + 1;
            }
        }
      }
      hs++;
    } while (hs < 2 * K && (!(hs & 1) || steps[4 * (long long)(hs >> 1) + 3] == dt1));
  }

#pragma unroll
  for (int k = 0; k < C; k++)
    if (lo + k < n) {
      const int i = off + lo + k;
      vm[i] = V[k];
#pragma unroll
      for (int q = 0; q < M::NS - 1; q++) gates[(long long)q * fb.gate_stride + i] = g[k][q];
      // the last check's Vm is the launch's final Vm
      if (spk.enabled) spk.vm_prev[i] = V[k];
    }
}

// one workgroup per fibre; its threads take as many nodes each as the fibre needs
template <class M, class G, class E, int T, int CMAX, bool TAPE>
__global__ __launch_bounds__(T, 2) void k_fibre(
    DevFibers fb, FibreStim st, double *__restrict__ vm, G *__restrict__ gates, const double *__restrict__ steps, int K,
    int n0D, int ie, const int *__restrict__ order, DevSpikes spk, DevTrace tr) {
  extern __shared__ double sh[];
  if (TAPE && tr.raise_priority) __builtin_amdgcn_s_setprio(2);
  const int f = __builtin_amdgcn_readfirstlane(order[blockIdx.x]);
  const int off = fb.fiber_off[f];
  const int n = fb.fiber_off[f + 1] - off;
  with_chunk_rows<CMAX>((n + T - 1) / T, [&](auto c_) {
    fibre_steps<M, G, E, T, decltype(c_)::value, TAPE>(fb, st, vm, gates, steps, K, n0D, ie, spk, tr, f, off, n, sh);
  });
}

}  // namespace fms
