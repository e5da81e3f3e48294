// berm_device.h -- block bodies of the frozen-strategy Bermudan swaption
// price and pathwise adjoint (the forward with checkpoints and the reverse
// sweep), shared by the single-product and batched kernels and the
// persistent portfolio kernel.
#pragma once

#include "lmm_step.h"

namespace koo {
namespace {

using namespace lmm;

constexpr int kMaxBermDates = 40;
struct BermArgs {
  int E, itm_only, last;
  signed char e_of_step[kMaxRates];  // exercise index of each step, -1 if none
  float sh[kMaxBermDates][2], sc[kMaxBermDates][2];
};

// Coefficients of the frozen strategy, date ei, function j, as FP32: from
// FP64 device memory (uniform addresses: scalar loads) or from an FP32 table.
struct CoefGlobal {
  const double* __restrict__ c;
  __device__ float operator()(int ei, int j) const { return static_cast<float>(c[6 * ei + j]); }
};
struct CoefTable {
  const float* t;
  __device__ float operator()(int ei, int j) const { return t[6 * ei + j]; }
};

// One block of the forward: paths [block * BD, ...) of product m.  tab: the step
// table (scalar loads).  Own: the blocks form one in LDS behind the states, and
// the first leaves it at `tab` if there is one.  Agent (the persistent kernel):
// the block's price partial is stored agent-coherent.
// The checkpoint rows are SweepPlan's, the 1/B row of the states at S1 holding
// the number of steps the wavefront ran (as float) in its place.
template <int F, int BD, int U, bool Agent = false, bool Own = Agent, class Coef>
__device__ __forceinline__ void berm_fwd_block(const Model& m, const BermArgs& b, const Coef& cf,
                                               float* __restrict__ tab,
                                               float* __restrict__ ckpt, float* __restrict__ lamt,
                                               int* __restrict__ tau_out,
                                               float* __restrict__ vout,
                                               double* __restrict__ part, int block) {
  extern __shared__ float lds[];
  const BlockPaths bp(m.P, block, BD);
  const int N = m.N;
  const bool valid = static_cast<int>(threadIdx.x) < bp.n;
  const size_t p = bp.p0 + threadIdx.x;
  const LaneRows<BD> X{lds + threadIdx.x};
  float* ltab = lds + static_cast<size_t>(N) * BD;
  if (Own) fill_step_table<F>(m, ltab);
  for (int r = 0; r < N; ++r) X.set(r, 0.0f);
  if (Own) __syncthreads();
  if (Own && tab && block == 0)
    for (int i = threadIdx.x; i < static_cast<int>(step_table_floats(N)); i += BD) tab[i] = ltab[i];
  const auto ctab = [&]() {
    if constexpr (Own) return static_cast<const float*>(ltab);
    else return cmem(tab);
  }();
  float invB = 1.0f, V = 0.0f;
  int tau = -1;
  bool done = !valid;
  auto row = [&](int r) { return ckpt + static_cast<size_t>(r) * bp.P; };
  int seg_step = m.S1, seg = 0;  // the next step whose states are kept
  auto keep_states = [&](int s) {
    const int lo = seg == 0 ? 0 : s;
    dump_states(bp, X,
                row(seg == 0 ? sweep_state_row(F, m.S1)
                             : sweep_segment_row(N, F, m.S1, m.L, seg)),
                lo, N);
    ++seg;
    seg_step += m.L;
  };
  auto load = [&](int r) { return X.get(r); };
  float zn[F];
  load_z<F>(m, bp, 0, zn);
  Ahead<F, U> ahead;
  pc_fetch<F, U>(ahead, m, 0, ctab, load);
  // last step: none from when all of the wavefront's paths have exercised (a
  // scalar in the loop's one exit, so what the loop carries stays uniform)
  const auto last_step = [&](int last) {
    return __builtin_amdgcn_readfirstlane(__builtin_amdgcn_ballot_w64(!done) != 0 ? last : -1);
  };
  int steps = 0;  // run so far
  for (int s = 0, last = last_step(b.last); s <= last; ++s, last = last_step(last)) {
    if (s == seg_step) keep_states(s);
    float z[F], y[F], d[F];
#pragma unroll
    for (int f = 0; f < F; ++f) z[f] = zn[f];
    load_z<F>(m, bp, min(s + 1, N - 1), zn);
    const float xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load,
                                   [&](int r, float x) { X.set(r, x); });
    steps = s + 1;
    if (s + 1 < N) pc_fetch<F, U>(ahead, m, s + 1, ctab, load);
    if (s < m.S1) store_sums<F>(bp, row(2 * F * s), y, d);
    const float fs = fmaf(start_level(m, s), fast_exp2(xs), -m.disp[s]);
    const int ei = b.e_of_step[s];
    if (ei >= 0) {  // uniform: done lanes walk along
      float disc = 1.0f, ann = 0.0f, flt = 0.0f;
      walk_curve<U, false>(m, s, X, [&](int, float, float fr, float tr) {
        disc *= fast_rcp(1.0f + tr * fr);
        ann += tr * disc;
        flt += tr * fr * disc;
      });
      const float sr = flt / ann;
      const float ev = (sr - m.strike) * ann;
      const float x0 = (sr - b.sh[ei][0]) * b.sc[ei][0];
      const float x1 = (fs - b.sh[ei][1]) * b.sc[ei][1];
      const float cont = cf(ei, 0) + cf(ei, 1) * x0 + cf(ei, 2) * x1 + cf(ei, 3) * x0 * x0 +
                         cf(ei, 4) * x0 * x1 + cf(ei, 5) * x1 * x1;
      const float evp = ev > 0.0f ? ev : 0.0f;
      const bool allowed = !b.itm_only || evp > 0.0f;
      const bool now = !done && allowed && cont - evp < 0.0f;
      if (__any(now)) {
        done = done || now;
        tau = now ? s : tau;
        V = now ? evp * invB : V;
        // payoff adjoint on the end-of-step states r >= s (the other lanes'
        // stores are out of their buffer's range)
        const int byte = now ? static_cast<int>(4 * threadIdx.x) : -4;
        float Pr = disc, Q = 0.0f;  // P_{r+1}, sum_{m>r} tau_{m-1} P_m
        walk_curve<U, true>(m, s, X, [&](int r, float x, float fr, float tr) {
          const float g = tr * fast_rcp(1.0f + tr * fr);
          Q += tr * Pr;
          PathRow row = bp.row(lamt, r);
          row.byte = byte;
          row.store(ev > 0.0f ? g * (disc + m.strike * Q) * invB * x * kLn2 : 0.0f);
          Pr *= 1.0f + tr * fr;
        });
      }
    }
    invB *= fast_rcp(1.0f + m.taus[s] * fs);
  }
  if (seg == 0) keep_states(steps);  // stopped before step S1
  bp.row(row(sweep_state_row(F, m.S1)), N).store(static_cast<float>(steps));
  if (valid) {
    tau_out[p] = tau;
    vout[p] = V;
  }
  const double sum = wave_sum_f64(valid ? static_cast<double>(V) : 0.0);
  if ((threadIdx.x & 63) == 0)
    put_partial<Agent>(part, wave_count(m.P), wave_index<BD>(block), 0, sum);
}

// One block of the backward (paths [block * BD, ...)).  LDS: the state adjoints
// and the states, 2N rows of lanes.  Agent (the persistent kernel): the
// partials stored agent-coherent; the step table in LDS behind the adjoints,
// and the states in place in the rows that the forward kept them in (the next
// run's forward writes those again), so that three blocks fit a CU as in its
// other phases.
template <int F, int BD, int U, bool Agent = false>
__device__ __forceinline__ void berm_bwd_block(const Model& m, const float* __restrict__ vols,
                                               const float* __restrict__ tab,
                                               float* __restrict__ ckpt,
                                               const float* __restrict__ lamt,
                                               const int* __restrict__ tau_in,
                                               const float* __restrict__ vin,
                                               float* __restrict__ scratch,
                                               double* __restrict__ part, int block) {
  extern __shared__ float lds[];
  const BlockPaths bp(m.P, block, BD);
  const int N = m.N;
  const bool valid = static_cast<int>(threadIdx.x) < bp.n;
  const size_t p = bp.p0 + threadIdx.x;
  const LaneRows<BD> lam{lds + threadIdx.x};
  float* ltab = lds + static_cast<size_t>(N) * BD;
  if (Agent) fill_step_table<F>(m, ltab);
  for (int r = 0; r < N; ++r) lam.set(r, 0.0f);
  if (Agent) __syncthreads();
  const auto ctab = [&]() {
    if constexpr (Agent) return static_cast<const float*>(ltab);
    else return cmem(tab);
  }();
  VegaSums<kVegaTiles<BD>> vegas;
  vegas.clear();

  const int tau = valid ? tau_in[p] : -1;
  const float V = valid ? vin[p] : 0.0f;
  auto row = [&](int r) { return ckpt + static_cast<size_t>(r) * bp.P; };
  float* states = row(sweep_state_row(F, m.S1));
  // the states, from their rows at `rows` (rates lo..N-1)
  auto begin_states = [&](float* rows, int lo) {
    if constexpr (Agent) {
      return GlobalRows{bp, rows - static_cast<size_t>(lo) * bp.P};
    } else {
      const LaneRows<BD> X{lds + N * BD + threadIdx.x};
      load_states(bp, X, rows, lo, N);
      return X;
    }
  };
  // The steps the wavefront's forward ran, which the kept states are after: a
  // scalar, so that the loops below and their addresses are uniform.  (Lanes
  // past the last path read 0; a wavefront of such lanes does nothing.)
  const int top = __builtin_amdgcn_readfirstlane(static_cast<int>(bp.row(states, N).load()));
  // Lanes past the last path have no exercise step: their adjoints stay zero.
  NonFinite bad;
  auto seed = [&](int s) {
    if (s == tau)  // the payoff adjoint recorded at exercise
      for (int r = s; r < N; ++r) {
        float lp = bp.row(lamt, r).load();
        bad.take(lp, r);
        lam.set(r, lp);
      }
  };
  auto fixing = [&](int s, float& lp, float x) {
    // the fixing inside B_tau
    const float xs = start_level(m, s) * fast_exp2(x);
    const float ti = m.taus[s] * fast_rcp(1.0f + m.taus[s] * (xs - m.disp[s]));
    if (s < tau) lp -= ti * V * xs * kLn2;
    bad.take(lp, s);
  };
  // The steps from S1 on: each segment run again, its sums to scratch, then
  // reversed.
  for (int seg = m.S1 < top ? (top - m.S1 - 1) / m.L : -1; seg >= 0; --seg) {
    const int s0 = m.S1 + seg * m.L, s1 = min(top, s0 + m.L);
    const auto X =
        seg == 0 ? begin_states(states, 0)  // the rates that have fixed come first
                 : begin_states(row(sweep_segment_row(N, F, m.S1, m.L, seg)), s0);
    auto load = [&](int r) { return X.get(r); };
    float zn[F];
    load_z<F>(m, bp, s0, zn);
    Ahead<F, U> ahead;
    pc_fetch<F, U>(ahead, m, s0, ctab, load);
    for (int s = s0; s < s1; ++s) {
      float z[F], y[F], d[F];
#pragma unroll
      for (int f = 0; f < F; ++f) z[f] = zn[f];
      load_z<F>(m, bp, min(s + 1, N - 1), zn);
      pc_step<F, U>(m, s, ctab, ahead, z, y, d, load, [&](int r, float x) { X.set(r, x); });
      if (s + 1 < s1) pc_fetch<F, U>(ahead, m, s + 1, ctab, load);
      store_sums<F>(bp, scratch + static_cast<size_t>(2 * F * (s - s0)) * bp.P, y, d);
    }
    reverse_steps<F, U>(m, bp, s1, s0, scratch, ctab, X, lam, seed, fixing, vegas);
  }
  // The steps whose sums the forward kept, from the states there or those that
  // segment 0 has gone back to (which are in place already).
  const auto X = [&]() {
    if constexpr (Agent) return GlobalRows{bp, states};
    else return LaneRows<BD>{lds + N * BD + threadIdx.x};
  }();
  if (!Agent && top <= m.S1) load_states(bp, X, states, 0, N);
  reverse_steps<F, U>(m, bp, min(top, m.S1), 0, ckpt, ctab, X, lam, seed, fixing, vegas);
  adjoint_sums<BD, Agent>(m, vols, lam, vegas, bad, part, block);
}

// Lanes per block of the single-product kernels (the batched and persistent
// ones run kAdjLanes).
int fwd_lanes(int paths, int N) {
  return N < kShortCurve || (N <= 2 * kAdjRates && paths >= 32768) ? kAdjLanes : 64;
}
int bwd_lanes(int paths, int N) {
  return N < kShortCurve || (N <= kAdjRates && paths >= 32768) ? kAdjLanes : 64;
}
// lds_table: the persistent kernel, which keeps the step table in LDS.
size_t rows_lds(int N, int rows, int lanes, bool lds_table) {
  return sizeof(float) *
         (static_cast<size_t>(rows) * lanes + (lds_table ? step_table_floats(N) : 0));
}

// Host checks and the strategy argument.
int check_berm(const char* who, int paths, int rates, int factors, int k) {
  if (paths < 1 || rates < 1 || rates > kMaxRates || factors < 1 || factors > kMaxFactors || k < 1)
    return set_error(KOO_ERR_INVALID,
                     "%s: need paths>=1, 1<=rates<=%d, 1<=factors<=%d, checkpoint_every>=1 "
                     "(got %d, %d, %d, %d)",
                     who, kMaxRates, kMaxFactors, paths, rates, factors, k);
  return KOO_OK;
}

// Host strategy -> kernel argument.
int make_berm_args(const char* who, int rates, int n_ex, const int* ex_steps,
                   const double* shift, const double* scale, int itm_only, BermArgs* b) {
  if (n_ex < 1 || n_ex > kMaxBermDates || !ex_steps)
    return set_error(KOO_ERR_INVALID, "%s: need 1<=exercise dates<=%d", who, kMaxBermDates);
  *b = BermArgs{};
  for (int s = 0; s < kMaxRates; ++s) b->e_of_step[s] = -1;
  for (int e = 0; e < n_ex; ++e) {
    const int s = ex_steps[e];
    if (s < 0 || s >= rates || (e > 0 && s <= ex_steps[e - 1]))
      return set_error(KOO_ERR_INVALID, "%s: exercise steps must increase within [0, %d)", who,
                       rates);
    b->e_of_step[s] = static_cast<signed char>(e);
    for (int i = 0; i < 2; ++i) {
      b->sh[e][i] = shift ? static_cast<float>(shift[2 * e + i]) : 0.0f;
      b->sc[e][i] = scale ? static_cast<float>(scale[2 * e + i]) : 1.0f;
    }
  }
  b->E = n_ex;
  b->itm_only = itm_only != 0;
  b->last = ex_steps[n_ex - 1];
  return KOO_OK;
}

}  // namespace
}  // namespace koo
