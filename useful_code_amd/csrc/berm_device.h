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

__device__ __forceinline__ int wave_max_int(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// Floats of a product's checkpoint buffer before the step table that the
// single-product and batched forwards copy behind them.
template <int F>
__device__ __forceinline__ size_t berm_ckpt_floats(const Model& m) {
  const size_t rows = m.k == 1 ? m.N + 1 + 2 * F : m.N + 1;
  return static_cast<size_t>((m.N + m.k - 1) / m.k) * rows * static_cast<size_t>(m.P);
}

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

// One block of the forward: paths [block * BD, ...) of product m.  Ctab: the
// step table behind the checkpoints (scalar loads), or the block's own copy in
// LDS behind its states (the persistent kernel, whose backward runs in the
// same launch).  Agent: the block's price partial stored agent-coherent (the
// persistent kernel).
template <int F, int BD, int U, bool Agent = false, class Coef>
__device__ __forceinline__ void berm_fwd_block(const Model& m, const BermArgs& b, const Coef& cf,
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
  if (Agent) fill_step_table<F>(m, ltab);
  for (int r = 0; r < N; ++r) X.set(r, 0.0f);
  if (Agent) __syncthreads();
  const auto ctab = [&]() {
    if constexpr (Agent) return static_cast<const float*>(ltab);
    else return cmem(ckpt + berm_ckpt_floats<F>(m));
  }();
  float invB = 1.0f, V = 0.0f;
  int tau = -1;
  bool done = !valid;
  const int rows = m.k == 1 ? N + 1 + 2 * F : N + 1;
  auto slot = [&](int s) { return ckpt + static_cast<size_t>(s / m.k) * rows * bp.P; };
  for (int r = 0; r < N; ++r) bp.row(slot(0), r).store(0.0f);
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
  for (int s = 0, last = last_step(b.last); s <= last; ++s, last = last_step(last)) {
    float z[F], y[F], d[F];
#pragma unroll
    for (int f = 0; f < F; ++f) z[f] = zn[f];
    load_z<F>(m, bp, min(s + 1, N - 1), zn);
    float xs;
    if (s + 1 < N && (s + 1) % m.k == 0) {
      const float* next = slot(s + 1);
      xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load, [&](int r, float x) {
        X.set(r, x);
        bp.row(next, r).store(x);
      });
    } else {
      xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load, [&](int r, float x) { X.set(r, x); });
    }
    if (s + 1 < N) pc_fetch<F, U>(ahead, m, s + 1, ctab, load);
    if (s % m.k == 0) {
      const float* c = slot(s) + static_cast<size_t>(N) * bp.P;
      bp.row(c).store(invB);
      if (m.k == 1) store_sums<F>(bp, c + bp.P, y, d);
    }
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
  if (valid) {
    tau_out[p] = tau;
    vout[p] = V;
  }
  // (the states are done with: their rows hold the wavefronts' sums)
  block_sum_to<Agent>(valid ? static_cast<double>(V) : 0.0, reinterpret_cast<double*>(lds),
                      part + block);
}

// One block of the backward (paths [block * BD, ...)).  Agent: the block's
// partials stored agent-coherent (persistent kernel).  LDS: the state adjoints
// [N][lanes], and the step table in the persistent kernel only (the others
// read the forward's behind the checkpoints through the scalar cache).
template <int F, int BD, int U, bool Agent = false>
__device__ __forceinline__ void berm_bwd_block(const Model& m, const float* __restrict__ vols,
                                               const float* __restrict__ ckpt,
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
    else return cmem(ckpt + berm_ckpt_floats<F>(m));
  }();
  VegaSums<kVegaTiles<BD>> vegas;
  vegas.clear();

  const int tau = valid ? tau_in[p] : -1;
  const float V = valid ? vin[p] : 0.0f;
  // The wavefront's last exercise step, made a scalar (the butterfly leaves
  // it in every lane) so the loops below and their addresses are uniform.
  const int s_top = __builtin_amdgcn_readfirstlane(wave_max_int(tau));
  const size_t slot = static_cast<size_t>(N + 1 + 2 * F) * bp.P;
  const bool every = m.k == 1;
  Ahead<F, U> ahead;
  for (int seg = s_top < 0 ? -1 : s_top / m.k; seg >= 0; --seg) {
    const int s0 = seg * m.k;
    const int s1 = min(s_top + 1, s0 + m.k);
    const float* ck = ckpt + static_cast<size_t>(seg) * (every ? slot : (N + 1) * bp.P);
    for (int s = s0; s < (every ? s0 : s1); ++s) {
      const int j = s - s0;
      const float* src = j == 0 ? ck : scratch + j * slot;
      float* cur = scratch + j * slot;
      float* dst = cur + slot;
      const bool keep = s + 1 < s1;
      float z[F], y[F], d[F];
      load_z<F>(m, bp, s, z);
      auto load = [&](int r) { return bp.row(src, r).load(); };
      if (j == 0) pc_fetch<F, U>(ahead, m, s, ctab, load);
      const float xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load, [&](int r, float x) {
        bp.row(dst, r, keep).store(x);
      });
      if (keep)
        pc_fetch<F, U>(ahead, m, s + 1, ctab, [&](int r) { return bp.row(dst, r).load(); });
      store_sums<F>(bp, cur + static_cast<size_t>(N + 1) * bp.P, y, d);
      if (keep) {
        const float fs = fmaf(start_level(m, s), fast_exp2(xs), -m.disp[s]);
        bp.row(dst, N).store(bp.row(src, N).load() * fast_rcp(1.0f + m.taus[s] * fs));
      }
    }
    for (int s = s1 - 1; s >= s0; --s) {
      const int j = s - s0;
      const float* src = j == 0 ? ck : scratch + j * slot;
      const float* sums = every ? ck : scratch + j * slot;
      if (s == tau)  // seed lambda with the payoff adjoint recorded at exercise
        for (int r = s; r < N; ++r) lam.set(r, bp.row(lamt, r).load());
      auto load = [&](int r) { return bp.row(src, r).load(); };
      reverse_fetch<F, U>(ahead, m, s, ctab, load, lam);
      float y[F], d[F];
      load_sums<F>(bp, sums + static_cast<size_t>(N + 1) * bp.P, y, d);
      // Lanes past the last path read zeros and have no exercise step: their
      // adjoints stay zero.
      reverse_step<F, U>(
          m, s, ctab, ahead, load, lam, y, d,
          [&](float& lp, float x) {
            // the fixing inside B_tau
            const float xs = start_level(m, s) * fast_exp2(x);
            const float ti = m.taus[s] * fast_rcp(1.0f + m.taus[s] * (xs - m.disp[s]));
            if (s < tau) lp -= ti * V * xs * kLn2;
          },
          vegas);
    }
  }
  adjoint_sums<BD, Agent>(m, vols, lds, vegas, part + static_cast<size_t>(block) * 2 * N);
}

// Blocks of 256 lanes, as the batched and persistent kernels run (the same
// sums bit for bit); of one wavefront for long curves, whose rows fill the LDS
// in smaller pieces.
int block_lanes(int N) { return N <= 45 ? 256 : 64; }
// lds_table: the persistent kernel, which keeps the step table in LDS.
size_t rows_lds(int N, int lanes, bool lds_table) {
  return sizeof(float) *
         (static_cast<size_t>(N) * lanes + (lds_table ? step_table_floats(N) : 0));
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
