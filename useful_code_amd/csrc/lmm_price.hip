// lmm_price.hip -- fused LMM pricing with pathwise adjoint Greeks, gfx950.
//
// Forward (k_price_fwd): one lane per path evolves the whole rate curve with
// the predictor-corrector log-Euler step of LMM_evolver_all.cu:571-742 (spot
// measure, displaced diffusion), prices the product on the fly and never
// writes the rate cube: its only HBM traffic is the bridged variates (S,F,P)
// and, when asked, what the reverse sweep needs (SweepPlan, lmm_step.h).
//
// Backward (k_price_bwd): one reverse sweep per path.  The steps are reversed
// one by one, rates in descending order, from each step's final sums y, d: the
// states go back with them, the sums are un-accumulated and their adjoints
// accumulated in registers.  Sums that the forward had no room for are run
// again from kept states, into a scratch buffer.  Deltas come from the adjoint
// of the initial states; vegas from sum_{s,f} Abar(s,r,f) A(s,r,f) / sigma_r,
// whose per-rate contraction needs only quantities the reverse step already
// has (no per-factor Abar is formed).
//
// The model's uniform data (pseudo-roots, step table, taus, displacements) is
// read with uniform addresses (scalar loads); the per-path state lives in LDS
// laid out [rate][lane] so wavefront accesses are conflict free; wavefronts'
// partial sums are formed in FP64 and a final single pass sums them with
// compensation.
//
// Both kernels issue vector instructions most of the time, so they got faster
// by having fewer: the step in the state's units (relative, base 2), the
// diffusion carried along with the predictor drift, buffer addressing, the vega
// sums on the matrix cores, and fewer steps run again (at 40 rates, 5 factors
// and k = 8 those of 300 of the 820 rate updates; all of them while each step's
// states were kept in scratch, 14.8 GB of traffic).  At 2^20 paths, 40 rates, 5
// factors and k = 8: forward with checkpoints 1250 -> 845 us, backward 3655 ->
// 2440 us; at k = 8 and 4096 paths 188 -> 107 and 535 -> 230 us; price of 2^17
// paths, 80 rates, 2 factors 1525 -> 365 us (its step table was in LDS and left
// room for three wavefronts per CU).
#include "lmm_step.h"

namespace koo {

namespace {

using namespace lmm;


// Caplet value at fixing, tau max(f-K,0)/(1+tau f), and its f-derivative.
__device__ __forceinline__ float caplet_value(float f, float tau, float K, float inv) {
  return f > K ? tau * (f - K) * inv : 0.0f;
}
__device__ __forceinline__ float caplet_deriv(float f, float tau, float K, float inv) {
  return f > K ? tau * (1.0f + tau * K) * inv * inv : 0.0f;
}

// The step table of the model (lmm_step.h), where the pricing kernels read it
// with scalar loads.  One lane per entry of the square.
template <int F>
__global__ void __launch_bounds__(256) k_step_table(KOO_MODEL_PARAMS, float* __restrict__ tab) {
  KOO_MODEL_LOCAL;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < m.N * m.N) put_step_entry<F>(m, q, tab);
}

// Forward: the state of every rate in LDS, the uniform data of a step through
// scalar registers (pc_step): 4F + 10 vector instructions a rate update.
template <int F, int BD, int U>
__global__ void __launch_bounds__(BD)
    k_price_fwd(KOO_MODEL_PARAMS, const float* __restrict__ tab, float* __restrict__ ckpt,
                double* __restrict__ part) {
  KOO_MODEL_LOCAL;
  extern __shared__ float lds[];
  const BlockPaths b(m.P, blockIdx.x, BD);
  const LaneRows<BD> X{lds + threadIdx.x};
  const int N = m.N;
  const c_cfloat ctab = cmem(tab);
  for (int r = 0; r < N; ++r) X.set(r, 0.0f);
  float invB = 1.0f, v = 0.0f, vc = 0.0f;
  auto row = [&](int r) { return ckpt + static_cast<size_t>(r) * b.P; };
  int seg_step = ckpt ? m.S1 : N + 1, seg = 0;  // the next step whose states are kept
  auto keep_states = [&](int s) {
    const float* rows = row(seg == 0 ? sweep_state_row(F, m.S1)
                                     : sweep_segment_row(N, F, m.S1, m.L, seg));
    const int lo = seg == 0 ? 0 : s;
    dump_states(b, X, rows, lo, N);
    b.row(rows, N - lo).store(invB);
    ++seg;
    seg_step += m.L;
  };
  auto load = [&](int r) { return X.get(r); };
  float zn[F];
  load_z<F>(m, b, 0, zn);
  Ahead<F, U> ahead;
  pc_fetch<F, U>(ahead, m, 0, ctab, load);
  for (int s = 0; s < N; ++s) {
    if (s == seg_step) keep_states(s);
    float z[F], y[F], d[F];
#pragma unroll
    for (int f = 0; f < F; ++f) z[f] = zn[f];
    load_z<F>(m, b, min(s + 1, N - 1), zn);
    const float xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load,
                                   [&](int r, float x) { X.set(r, x); });
    if (s + 1 < N) pc_fetch<F, U>(ahead, m, s + 1, ctab, load);
    if (ckpt && s < m.S1) store_sums<F>(b, row(2 * F * s), y, d);
    const float tau = m.taus[s];
    const float fs = fmaf(start_level(m, s), fast_exp2(xs), -m.disp[s]);
    const float inv = fast_rcp(1.0f + tau * fs);
    // Kahan-compensated path sum of the deflated caplet values.
    const float term = caplet_value(fs, tau, m.strike, inv) * invB - vc;
    const float sum = v + term;
    vc = (sum - v) - term;
    v = sum;
    invB *= inv;
  }
  if (ckpt && seg == 0) keep_states(N);  // S1 == N
  const double sum = wave_sum_f64(static_cast<int>(threadIdx.x) < b.n ? static_cast<double>(v) : 0.0);
  if ((threadIdx.x & 63) == 0)
    put_partial<false>(part, wave_count(m.P), wave_index<BD>(blockIdx.x), 0, sum);
}

// Backward (SweepPlan, reverse_step).  LDS: the states and their adjoints, 2N
// rows of lanes: at 40 rates eight wavefronts per CU, which is enough for loops
// that touch no other memory.  W: wavefronts per SIMD that the registers are
// laid out for, so that single-wavefront blocks spread over the SIMDs.
template <int F, int BD, int U, int W>
__global__ void __launch_bounds__(BD) __attribute__((amdgpu_waves_per_eu(W, W)))
    k_price_bwd(KOO_MODEL_PARAMS, const float* __restrict__ vols, const float* __restrict__ ckpt,
                const float* __restrict__ tab, float* __restrict__ scratch,
                double* __restrict__ part) {
  KOO_MODEL_LOCAL;
  extern __shared__ float lds[];
  const BlockPaths b(m.P, blockIdx.x, BD);
  const int N = m.N;
  const c_cfloat ctab = cmem(tab);
  const LaneRows<BD> lam{lds + threadIdx.x};
  const LaneRows<BD> X{lds + N * BD + threadIdx.x};
  VegaSums<kVegaTiles<BD>> vegas;
  vegas.clear();
  for (int r = 0; r < N; ++r) lam.set(r, 0.0f);

  auto row = [&](int r) { return ckpt + static_cast<size_t>(r) * b.P; };
  float tail = 0.0f, invB = 0.0f;  // invB: 1/B after the step being reversed
  auto fixing = [&](int s, float& lp, float x) {
    // The rate fixing at the end of this step: caplet value and the numeraire
    // it enters for later fixings.  (Lanes past the last path read 1/B = 0,
    // so their adjoints stay zero.)
    const float tau = m.taus[s];
    const float xs = start_level(m, s) * fast_exp2(x);
    const float fs = xs - m.disp[s];
    const float grow = 1.0f + tau * fs, inv = fast_rcp(grow);
    invB *= grow;
    const float v = caplet_value(fs, tau, m.strike, inv);
    const float dv = caplet_deriv(fs, tau, m.strike, inv);
    lp = fmaf(dv * invB - tau * inv * tail, kLn2 * xs, lp);
    tail += v * invB;
  };
  auto nothing = [](int) {};
  // The steps from S1 on: each segment run again, its sums to scratch, then
  // reversed.
  for (int seg = m.S1 < N ? (N - m.S1 - 1) / m.L : -1; seg >= 0; --seg) {
    const int s0 = m.S1 + seg * m.L, s1 = min(N, s0 + m.L);
    const float* rows = row(seg == 0 ? sweep_state_row(F, m.S1)
                                     : sweep_segment_row(N, F, m.S1, m.L, seg));
    if (seg == 0) rows += static_cast<size_t>(s0) * b.P;  // the rates that have fixed come first
    load_states(b, X, rows, s0, N);
    invB = b.row(rows, N - s0).load();
    auto load = [&](int r) { return X.get(r); };
    float zn[F];
    load_z<F>(m, b, s0, zn);
    Ahead<F, U> ahead;
    pc_fetch<F, U>(ahead, m, s0, ctab, load);
    for (int s = s0; s < s1; ++s) {
      float z[F], y[F], d[F];
#pragma unroll
      for (int f = 0; f < F; ++f) z[f] = zn[f];
      load_z<F>(m, b, min(s + 1, N - 1), zn);
      const float xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load,
                                     [&](int r, float x) { X.set(r, x); });
      if (s + 1 < s1) pc_fetch<F, U>(ahead, m, s + 1, ctab, load);
      store_sums<F>(b, scratch + static_cast<size_t>(2 * F * (s - s0)) * b.P, y, d);
      const float fs = fmaf(start_level(m, s), fast_exp2(xs), -m.disp[s]);
      invB *= fast_rcp(1.0f + m.taus[s] * fs);
    }
    reverse_steps<F, U>(m, b, s1, s0, scratch, ctab, X, lam, nothing, fixing, vegas);
  }
  // The steps whose sums the forward kept.
  if (m.S1 > 0) {
    const float* rows = row(sweep_state_row(F, m.S1));
    load_states(b, X, rows, 0, N);
    invB = b.row(rows, N).load();
    reverse_steps<F, U>(m, b, m.S1, 0, ckpt, ctab, X, lam, nothing, fixing, vegas);
  }
  adjoint_sums<BD>(m, vols, lam, vegas, part, blockIdx.x);
}

int fwd_lanes(int paths, int N) {
  return N >= kShortCurve && N <= 2 * kAdjRates && paths >= 32768 ? kAdjLanes : 64;
}
int bwd_lanes(int paths, int N) {
  return N >= kShortCurve && N <= kAdjRates && paths >= 32768 ? kAdjLanes : 64;
}
size_t rows_lds(int rows, int lanes) { return sizeof(float) * static_cast<size_t>(rows) * lanes; }
// Doubles of the partials before the step table of a forward without
// checkpoints.
size_t partial_doubles(int paths, int N) { return static_cast<size_t>(wave_count(paths)) * 2 * N; }

int check_model(const char* who, int paths, int rates, int factors, int k, int product) {
  if (paths < 1 || rates < 1 || rates > kMaxRates || factors < 1 || factors > kMaxFactors || k < 1)
    return set_error(KOO_ERR_INVALID,
                     "%s: need paths>=1, 1<=rates<=%d, 1<=factors<=%d, checkpoint_every>=1 "
                     "(got %d, %d, %d, %d)",
                     who, kMaxRates, kMaxFactors, paths, rates, factors, k);
  if (product != KOO_PRODUCT_CAPLETS)
    return set_error(KOO_ERR_INVALID, "%s: unknown product %d", who, product);
  return KOO_OK;
}

}  // namespace
}  // namespace koo

using namespace koo;

extern "C" int lmm_price_workspace(int paths, int rates, int factors, int checkpoint_every,
                                   size_t* checkpoint_bytes, size_t* scratch_bytes,
                                   size_t* partial_bytes) {
  if (int e = check_model("lmm_price_workspace", paths, rates, factors, checkpoint_every,
                          KOO_PRODUCT_CAPLETS))
    return e;
  const size_t P = static_cast<size_t>(paths);
  const int k = checkpoint_every;
  if (checkpoint_bytes)
    *checkpoint_bytes =
        sizeof(float) * (ckpt_rows(rates, factors, k) * P + step_table_floats(rates));
  // k == 1 needs no recompute scratch; one float keeps the pointer non-null.
  if (scratch_bytes)
    *scratch_bytes = sizeof(float) * (k == 1 ? 1 : scratch_rows(rates, factors, k) * P);
  if (partial_bytes)
    *partial_bytes = sizeof(double) * partial_doubles(paths, rates) +
                     sizeof(float) * step_table_floats(rates);
  return KOO_OK;
}

extern "C" int lmm_price_fwd(int paths, int rates, int factors, int checkpoint_every,
                             const float* variates, const float* initial_rates, const float* taus,
                             const float* displacements, const float* pseudo_roots, int product,
                             const float* product_aux, float* checkpoints, double* partials,
                             double* price_out, void* stream) {
  if (int e = check_model("lmm_price_fwd", paths, rates, factors, checkpoint_every, product))
    return e;
  if (!variates || !initial_rates || !taus || !displacements || !pseudo_roots || !product_aux ||
      !partials || !price_out)
    return set_error(KOO_ERR_INVALID, "lmm_price_fwd: null pointer");
  const float strike = product_aux[0];
  const SweepPlan plan = sweep_plan(rates, factors, checkpoint_every);
  Model m{variates, cmem(initial_rates), cmem(taus), cmem(displacements), cmem(pseudo_roots),
          strike, paths, rates, plan.S1, plan.L};
  const int threads = fwd_lanes(paths, rates);
  const int blocks = (paths + threads - 1) / threads;
  const size_t lds = rows_lds(rates, threads);
  float* tab = checkpoints
                   ? checkpoints + static_cast<size_t>(ckpt_rows(rates, factors, checkpoint_every)) *
                                       paths
                   : reinterpret_cast<float*>(partials + partial_doubles(paths, rates));
  hipStream_t st = as_stream(stream);
  switch (factors) {
#define KOO_FWD(F, BD, U)                                                                        \
  hipLaunchKernelGGL((k_price_fwd<F, BD, U>), dim3(blocks), dim3(BD), lds, st, m.z, m.f0,        \
                     m.taus, m.disp, m.A, m.strike, m.P, m.N, m.S1, m.L, tab, checkpoints, partials)
#define KOO_CASE(F)                                                                              \
  case F:                                                                                        \
    hipLaunchKernelGGL(k_step_table<F>, dim3((rates * rates + 255) / 256), dim3(256), 0, st,     \
                       m.z, m.f0, m.taus, m.disp, m.A, m.strike, m.P, m.N, m.S1, m.L, tab);            \
    if (threads == kAdjLanes)                                                                          \
      KOO_FWD(F, kAdjLanes, kWindow<F>);                                                               \
    else if (rates >= kShortCurve)                                                               \
      KOO_FWD(F, 64, kWindow<F>);                                                                \
    else                                                                                         \
      KOO_FWD(F, 64, 1);                                                                         \
    break;
    KOO_CASE(1) KOO_CASE(2) KOO_CASE(3) KOO_CASE(4) KOO_CASE(5) KOO_CASE(6) KOO_CASE(7)
    KOO_CASE(8)
#undef KOO_CASE
#undef KOO_FWD
  }
  hipLaunchKernelGGL(k_finalize_rows, dim3(1), dim3(finalize_lanes(wave_count(paths))), 0, st,
                     partials, wave_count(paths), 1.0 / static_cast<double>(paths), price_out);
  return check_launch("lmm_price_fwd");
}

extern "C" int lmm_price_bwd(int paths, int rates, int factors, int checkpoint_every,
                             const float* variates, const float* initial_rates, const float* taus,
                             const float* displacements, const float* pseudo_roots,
                             const float* vols, int product, const float* product_aux,
                             const float* checkpoints, float* segment_scratch, double* partials,
                             double* greeks_out, void* stream) {
  if (int e = check_model("lmm_price_bwd", paths, rates, factors, checkpoint_every, product))
    return e;
  if (!variates || !initial_rates || !taus || !displacements || !pseudo_roots || !vols ||
      !product_aux || !checkpoints || !segment_scratch || !partials || !greeks_out)
    return set_error(KOO_ERR_INVALID, "lmm_price_bwd: null pointer");
  const float strike = product_aux[0];
  const SweepPlan plan = sweep_plan(rates, factors, checkpoint_every);
  Model m{variates, cmem(initial_rates), cmem(taus), cmem(displacements), cmem(pseudo_roots),
          strike, paths, rates, plan.S1, plan.L};
  const int threads = bwd_lanes(paths, rates);
  const int blocks = (paths + threads - 1) / threads;
  const size_t lds = rows_lds(2 * rates, threads);
  const float* tab =
      checkpoints + static_cast<size_t>(ckpt_rows(rates, factors, checkpoint_every)) * paths;
  hipStream_t st = as_stream(stream);
  switch (factors) {
#define KOO_BWD(F, BD, U, W)                                                                     \
  hipLaunchKernelGGL((k_price_bwd<F, BD, U, W>), dim3(blocks), dim3(BD), lds, st, m.z, m.f0,     \
                     m.taus, m.disp, m.A, m.strike, m.P, m.N, m.S1, m.L, vols, checkpoints, tab,       \
                     segment_scratch, partials)
#define KOO_CASE(F)                                                                              \
  case F:                                                                                        \
    if (threads == kAdjLanes)                                                                    \
      KOO_BWD(F, kAdjLanes, kWindow<F>, 2);                                                      \
    else if (rates > 64)                                                                         \
      KOO_BWD(F, 64, kWindow<F>, 1);                                                             \
    else if (rates >= kShortCurve)                                                               \
      KOO_BWD(F, 64, kWindow<F>, 2);                                                             \
    else                                                                                         \
      KOO_BWD(F, 64, 1, 2);                                                                      \
    break;
    KOO_CASE(1) KOO_CASE(2) KOO_CASE(3) KOO_CASE(4) KOO_CASE(5) KOO_CASE(6) KOO_CASE(7)
    KOO_CASE(8)
#undef KOO_CASE
#undef KOO_BWD
  }
  hipLaunchKernelGGL(k_finalize_rows, dim3(2 * rates), dim3(finalize_lanes(wave_count(paths))), 0,
                     st, partials, wave_count(paths), 1.0 / static_cast<double>(paths), greeks_out);
  return check_launch("lmm_price_bwd");
}
