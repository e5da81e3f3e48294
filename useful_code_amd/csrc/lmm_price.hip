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
// Few paths take the form with a path's rates across the lanes instead
// (lmm_across.h; k_price_fwd_across, k_price_bwd_across): it keeps nothing
// between forward and backward, which runs the steps again.
//
// Both kernels issue vector instructions most of the time, so they got faster
// by having fewer: the step in the state's units (relative, base 2), the
// diffusion carried along with the predictor drift, buffer addressing, the vega
// sums on the matrix cores, and fewer steps run again (at 40 rates, 5 factors
// and k = 8 those of 300 of the 820 rate updates; all of them while each step's
// states were kept in scratch, 14.8 GB of traffic).  At 2^20 paths, 40 rates, 5
// factors and k = 8: forward with checkpoints 1250 -> 850 us, backward 3655 ->
// 2500 us (up to 2700 where the card has clocked down); at k = 8 and 4096 paths
// 188 -> 107 and 535 -> 230 us, 51 and 107 with the rates across the lanes; price
// of 2^17 paths, 80 rates, 2 factors 1525 -> 365 us (its step table was in LDS
// and left room for three wavefronts per CU).  Greeks beyond 40 rates run
// single-wavefront blocks in the backward, three to seven to a CU: 2^17 paths x 5
// factors, k = 8, forward and backward 46 rates 1117 -> 868 us, 60 rates 2223 ->
// 1313, 90 rates 9300 -> 3529.
#include <algorithm>

#include "lmm_across.h"

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
// scalar registers (pc_step): 4F + 10 vector instructions a rate update.  Own:
// the blocks form the step table in LDS and the first leaves it at `tab`.
template <int F, int BD, int U, bool Own>
__global__ void __launch_bounds__(BD)
    k_price_fwd(KOO_MODEL_PARAMS, float* __restrict__ tab, float* __restrict__ ckpt,
                double* __restrict__ part) {
  KOO_MODEL_LOCAL;
  extern __shared__ float lds[];
  const BlockPaths b(m.P, blockIdx.x, BD);
  const LaneRows<BD> X{lds + threadIdx.x};
  const int N = m.N;
  const auto ctab = [&]() {
    if constexpr (Own) return static_cast<const float*>(lds + N * BD);
    else return cmem(tab);
  }();
  if (Own) {
    fill_step_table<F>(m, lds + N * BD);
    __syncthreads();
    if (ckpt && blockIdx.x == 0)
      for (int i = threadIdx.x; i < static_cast<int>(step_table_floats(N)); i += BD)
        tab[i] = lds[N * BD + i];
  }
  for (int r = 0; r < N; ++r) X.set(r, 0.0f);
  Deflator B;
  float v = 0.0f, vc = 0.0f;
  auto row = [&](int r) { return ckpt + static_cast<size_t>(r) * b.P; };
  int seg_step = ckpt ? m.S1 : N + 1, seg = 0;  // the next step whose states are kept
  auto keep_states = [&](int s) {
    const float* rows = row(seg == 0 ? sweep_state_row(F, m.S1)
                                     : sweep_segment_row(N, F, m.S1, m.L, seg));
    const int lo = seg == 0 ? 0 : s;
    dump_states(b, X, rows, lo, N);
    b.row(rows, N - lo).store(B.m);
    if (seg > 0 || sweep_exponent_row(N, m.S1)) b.row(rows, N - lo + 1).store(__int_as_float(B.e));
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
    const float term = caplet_value(fs, tau, m.strike, inv) * B.value() - vc;
    const float sum = v + term;
    vc = (sum - v) - term;
    v = sum;
    B.scale(inv);
  }
  if (ckpt && seg == 0) keep_states(N);  // S1 == N
  const double sum =
      wave_sum_f64(static_cast<int>(threadIdx.x) < b.n ? static_cast<double>(v) : 0.0);
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
  NonFinite bad;
  float tail = 0.0f;
  Deflator B;  // after the step being reversed
  auto load_deflator = [&](const float* rows, int r, bool exponent) {
    B.m = b.row(rows, r).load();
    B.e = exponent ? __float_as_int(b.row(rows, r + 1).load()) : 0;
  };
  auto fixing = [&](int s, float& lp, float x) {
    // The rate fixing at the end of this step: caplet value and the numeraire
    // it enters for later fixings.  (Lanes past the last path read 1/B = 0,
    // so their adjoints stay zero.)
    const float tau = m.taus[s];
    const float xs = start_level(m, s) * fast_exp2(x);
    const float fs = xs - m.disp[s];
    const float grow = 1.0f + tau * fs, inv = fast_rcp(grow);
    B.scale(grow);
    const float invB = B.value();
    const float v = caplet_value(fs, tau, m.strike, inv);
    const float dv = caplet_deriv(fs, tau, m.strike, inv);
    lp = fmaf(dv * invB - tau * inv * tail, kLn2 * xs, lp);
    bad.take(lp, s);
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
    load_deflator(rows, N - s0, seg > 0 || sweep_exponent_row(N, m.S1));
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
      B.scale(fast_rcp(1.0f + m.taus[s] * fs));
    }
    reverse_steps<F, U>(m, b, s1, s0, scratch, ctab, X, lam, nothing, fixing, vegas);
  }
  // The steps whose sums the forward kept.
  if (m.S1 > 0) {
    const float* rows = row(sweep_state_row(F, m.S1));
    load_states(b, X, rows, 0, N);
    load_deflator(rows, N, sweep_exponent_row(N, m.S1));
    reverse_steps<F, U>(m, b, m.S1, 0, ckpt, ctab, X, lam, nothing, fixing, vegas);
  }
  adjoint_sums<BD>(m, vols, lam, vegas, bad, part, blockIdx.x);
}

// Few paths: the rates of a path across W lanes (lmm_across.h).  Once the paths
// have fixed, every lane values its own caplet: 1/B as a product scan, and for
// the adjoint the value of the later caplets as a sum scan.
struct Fixing {
  float inv, before, v;  // 1 / (1 + tau f), 1/B before the step, deflated value
};
template <int W>
__device__ __forceinline__ Fixing across_fixing(const Model& m, const AcrossLane<W>& at, float x) {
  Fixing o{1.0f, 0.0f, 0.0f};
  float f = 0.0f, tau = 0.0f;
  if (at.live) {
    tau = m.taus[at.r];
    f = fmaf(start_level(m, at.r), fast_exp2(x), -m.disp[at.r]);
    o.inv = fast_rcp(1.0f + tau * f);
  }
  const float upto = __shfl_up(scan_mul<W>(o.inv), 1, W);
  o.before = at.r ? upto : 1.0f;
  if (at.live) o.v = caplet_value(f, tau, m.strike, o.inv) * o.before;
  return o;
}

template <int F, int W>
__global__ void __launch_bounds__(kAcrossLanes)
    k_price_fwd_across(KOO_MODEL_PARAMS, double* __restrict__ part) {
  KOO_MODEL_LOCAL;
  __shared__ double red[kAcrossLanes / 64];
  const AcrossLane<W> at(m, blockIdx.x);
  const float kr = at.rate ? drift_constant(m, at.r) : 1.0f;
  const float x = across_steps<F, W>(m, at, kr, [](int, float, float, float) {});
  block_sum_to(static_cast<double>(across_fixing<W>(m, at, x).v), red, part + blockIdx.x);
}

// The forward again with what the reverse needs in LDS, then the reverse.
template <int F, int W>
__global__ void __launch_bounds__(kAcrossLanes)
    k_price_bwd_across(KOO_MODEL_PARAMS, const float* __restrict__ vols,
                       double* __restrict__ part) {
  KOO_MODEL_LOCAL;
  extern __shared__ float lds[];
  const AcrossLane<W> at(m, blockIdx.x);
  const int N = m.N, path = static_cast<int>(threadIdx.x) / W, tri = across_tri(N);
  float* mine = lds + static_cast<size_t>(path) * 3 * tri;
  const float kr = at.rate ? drift_constant(m, at.r) : 1.0f;
  const float xf = across_steps<F, W>(m, at, kr, [&](int s, float x, float my, float md) {
    if (at.rate && at.r >= s) {
      float* o = mine + across_tri_row(N, s) + N - 1 - at.r;
      o[0] = x;
      o[tri] = my;
      o[2 * tri] = md;
    }
  });
  const Fixing fx = across_fixing<W>(m, at, xf);
  // from here the lane has rate r = N - 1 - (its place)
  const int l = at.r, r = max(N - 1 - l, 0);
  const bool rate = at.rate;
  const float x = __shfl(xf, r, W), inv = __shfl(fx.inv, r, W), before = __shfl(fx.before, r, W);
  const float v = __shfl(fx.v, r, W);
  const float above = __shfl_up(scan_add<W>(rate ? v : 0.0f), 1, W);
  float lam = 0.0f, krr = 1.0f;
  if (rate) krr = drift_constant(m, r);
  if (at.live) {
    const float tau = m.taus[r], xs = start_level(m, r) * fast_exp2(x);
    const float tail = l ? above : 0.0f;
    lam = (caplet_deriv(xs - m.disp[r], tau, m.strike, inv) * before - tau * inv * tail) *
          (kLn2 * xs);
  }
  __syncthreads();
  const float w = across_reverse<F, W>(m, rate ? r : -1, rate, krr, lam,
                                       [&](int s, float& xo, float& my, float& md) {
    const float* o = mine + min(across_tri_row(N, s) + l, tri - 1);
    xo = o[0];
    my = o[tri];
    md = o[2 * tri];
  });
  // the block's sums, FP64
  __syncthreads();
  float* sums = lds;  // [path][2][W]
  sums[(path * 2) * W + l] = lam;
  sums[(path * 2 + 1) * W + l] = w;
  __syncthreads();
  for (int t = threadIdx.x; t < 2 * N; t += kAcrossLanes) {
    const int which = t >= N, rr = which ? t - N : t;
    double sum = 0.0;
    for (int i = 0; i < kAcrossBlock<W>; ++i)
      sum += static_cast<double>(sums[(i * 2 + which) * W + N - 1 - rr]);
    part[static_cast<size_t>(t) * gridDim.x + blockIdx.x] =
        which ? sum / static_cast<double>(vols[rr])
              : sum * static_cast<double>(kLog2e) / static_cast<double>(start_level(m, rr));
  }
}

// Lanes per path of the across form, 0 for a path per lane.  The across form
// takes time with its wavefronts beyond the first thousand, the path per lane
// the same up to 2^15 paths; forward and backward together cross at about 10000
// wavefronts of 64-lane paths (40 rates, 5 factors: 158 us for 336 at 4096
// paths, 273 at 8192, 479 at 16384), 7500 of 32-lane ones (20 rates, 3 factors:
// 71 us for 100 at 8192 paths, 107 at 16384) and 5500 of 16-lane ones (16
// rates, 5 factors: 76 us for 93 at 16384 paths, 116 at 32768).  With more dead
// lanes the limits still hold: 33 rates, 5 factors 197 for 235 us, 17 rates 81 for
// 96, 6 rates 29 for 32, 8 rates and 8 factors 44 each.  The price alone crosses
// near them too (40 rates 75 for 92 us, 17 rates 26 for 28), but for curves of up
// to 8 rates and 8 factors, where a path per lane takes 12.7 for 15.8 us at the
// limit: not worth a limit of its own.
int across_lanes(int paths, int N) {
  if (N < kShortCurve || N > 64) return 0;
  const int W = N <= 16 ? 16 : (N <= 32 ? 32 : 64);
  const int most = W == 16 ? 4096 : (W == 32 ? 6144 : 8192);  // wavefronts
  return paths <= most * (64 / W) ? W : 0;
}
size_t across_lds(int N, int W) {
  const size_t kept = sizeof(float) * (kAcrossLanes / W) * 3 * across_tri(N);
  return std::max(kept, sizeof(float) * 2 * kAcrossLanes);
}
int across_blocks(int paths, int W) { return (paths + kAcrossLanes / W - 1) / (kAcrossLanes / W); }

int fwd_lanes(int paths, int N) {
  return N >= kShortCurve && N <= 2 * kAdjRates && paths >= 32768 ? kAdjLanes : 64;
}
int bwd_lanes(int paths, int N) {
  return N >= kShortCurve && N <= kAdjRates && paths >= 32768 ? kAdjLanes : 64;
}
// Whether the forward's blocks form the step table, and not a launch before it:
// on short curves the launch is longer than what its scalar loads save (price of
// 16448 paths, 5 factors x 4 rates 14.1 us for 11.4, 8 factors x 8 rates 14.4 for
// 12.7; at 12 rates the table has 144 entries a block to form).
bool own_table(int rates, int lanes) { return rates < kShortCurve || (rates <= 8 && lanes == 64); }
size_t rows_lds(int rows, int lanes) { return sizeof(float) * static_cast<size_t>(rows) * lanes; }
// Doubles of the partials before the step table of a forward without
// checkpoints.
size_t partial_doubles(int paths, int N) {
  const int W = across_lanes(paths, N);
  const int columns = W ? std::max(across_blocks(paths, W), wave_count(paths)) : wave_count(paths);
  return static_cast<size_t>(columns) * 2 * N;
}

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

// KOO_W(F, W) for the factors and the lanes per path of the call.
#define KOO_ACROSS_CASE(F)        \
  case F:                         \
    if (W == 16) KOO_W(F, 16);    \
    else if (W == 32) KOO_W(F, 32); \
    else KOO_W(F, 64);            \
    break;
#define KOO_ACROSS_CASES                                                                    \
  switch (factors) {                                                                        \
    KOO_ACROSS_CASE(1) KOO_ACROSS_CASE(2) KOO_ACROSS_CASE(3) KOO_ACROSS_CASE(4)             \
    KOO_ACROSS_CASE(5) KOO_ACROSS_CASE(6) KOO_ACROSS_CASE(7) KOO_ACROSS_CASE(8)             \
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
  const bool own = own_table(rates, threads);
  const size_t lds =
      rows_lds(rates, threads) + (own ? sizeof(float) * step_table_floats(rates) : 0);
  const size_t kept = static_cast<size_t>(ckpt_rows(rates, factors, checkpoint_every)) * paths;
  float* tab = checkpoints ? checkpoints + kept
                           : reinterpret_cast<float*>(partials + partial_doubles(paths, rates));
  hipStream_t st = as_stream(stream);
  if (const int W = across_lanes(paths, rates)) {
    const int nb = across_blocks(paths, W);
#define KOO_W(F, W)                                                                              \
  hipLaunchKernelGGL((k_price_fwd_across<F, W>), dim3(nb), dim3(kAcrossLanes), 0, st, m.z, m.f0, \
                     m.taus, m.disp, m.A, m.strike, m.P, m.N, m.S1, m.L, partials)
    KOO_ACROSS_CASES
#undef KOO_W
    hipLaunchKernelGGL(k_finalize_rows, dim3(1), dim3(finalize_lanes(nb)), 0, st, partials, nb,
                       1.0 / static_cast<double>(paths), price_out);
    return check_launch("lmm_price_fwd");
  }
  switch (factors) {
#define KOO_FWD(F, BD, U, Own)                                                                   \
  hipLaunchKernelGGL((k_price_fwd<F, BD, U, Own>), dim3(blocks), dim3(BD), lds, st, m.z, m.f0,   \
                     m.taus, m.disp, m.A, m.strike, m.P, m.N, m.S1, m.L, tab, checkpoints,       \
                     partials)
#define KOO_CASE(F)                                                                              \
  case F:                                                                                        \
    if (!own)                                                                                    \
      hipLaunchKernelGGL(k_step_table<F>, dim3((rates * rates + 255) / 256), dim3(256), 0, st,   \
                         m.z, m.f0, m.taus, m.disp, m.A, m.strike, m.P, m.N, m.S1, m.L, tab);    \
    if (threads == kAdjLanes)                                                                    \
      KOO_FWD(F, kAdjLanes, kWindow<F>, false);                                                  \
    else if (rates < kShortCurve)                                                                \
      KOO_FWD(F, 64, 1, true);                                                                   \
    else if (own)                                                                                \
      KOO_FWD(F, 64, kWindow<F>, true);                                                          \
    else                                                                                         \
      KOO_FWD(F, 64, kWindow<F>, false);                                                         \
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
  if (const int W = across_lanes(paths, rates)) {
    const int nb = across_blocks(paths, W);
    const size_t bytes = across_lds(rates, W);
#define KOO_W(F, W)                                                                              \
  hipLaunchKernelGGL((k_price_bwd_across<F, W>), dim3(nb), dim3(kAcrossLanes), bytes, st, m.z,   \
                     m.f0, m.taus, m.disp, m.A, m.strike, m.P, m.N, m.S1, m.L, vols, partials)
    KOO_ACROSS_CASES
#undef KOO_W
    hipLaunchKernelGGL(k_finalize_rows, dim3(2 * rates), dim3(finalize_lanes(nb)), 0, st, partials,
                       nb, 1.0 / static_cast<double>(paths), greeks_out);
    return check_launch("lmm_price_bwd");
  }
  switch (factors) {
#define KOO_BWD(F, BD, U, W)                                                                     \
  hipLaunchKernelGGL((k_price_bwd<F, BD, U, W>), dim3(blocks), dim3(BD), lds, st, m.z, m.f0,     \
                     m.taus, m.disp, m.A, m.strike, m.P, m.N, m.S1, m.L, vols, checkpoints, tab, \
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
