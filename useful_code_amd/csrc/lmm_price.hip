// lmm_price.hip -- fused LMM pricing with pathwise adjoint Greeks, gfx950.
//
// Forward (k_price_fwd): one lane per path evolves the whole rate curve with
// the predictor-corrector log-Euler step of LMM_evolver_all.cu:571-742 (spot
// measure, displaced diffusion), prices the product on the fly and never
// writes the rate cube: its only HBM traffic is the bridged variates (S,F,P)
// and, when asked, one checkpoint of the state every k steps.
//
// Backward (k_price_bwd): one reverse sweep per path.  For each checkpoint
// segment, last first, the k steps are recomputed from the checkpoint and
// each step's start state and final sums y, d (lmm_step.h) are kept in a
// scratch buffer; then the steps are reversed one by one, rates in descending
// order, with the sums un-accumulated and their adjoints accumulated in
// registers.  Deltas come from the adjoint of the initial states; vegas from
// sum_{s,f} Abar(s,r,f) A(s,r,f) / sigma_r, whose per-rate contraction needs
// only quantities the reverse step already has (no per-factor Abar is formed).
//
// The model's uniform data (pseudo-roots, step table, taus, displacements) is
// read with uniform addresses (scalar loads); the per-path state lives in LDS
// laid out [rate][lane] so wavefront accesses are conflict free; block partial
// sums are formed in FP64 and a final single pass sums them with compensation.
//
// Both kernels issue vector instructions most of the time, so they got faster
// by having fewer: the step in the state's units (relative, base 2), the
// diffusion carried along with the predictor drift, buffer addressing and the
// vega sums on the matrix cores.  At 2^20 paths, 40 rates, 5 factors and k = 8:
// forward with checkpoints 1372 -> 1025 us, backward 3891 -> 3616 us; price of
// 2^17 paths, 80 rates, 2 factors 1540 -> 520 us (its step table was in LDS and
// left room for three wavefronts per CU).
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
  // Checkpoint of step s (s % k == 0): start states, row N: 1/B.  With k == 1
  // every step is one and also keeps its final sums (rows N+1..N+2F), so the
  // reverse sweep needs no recomputation.  The states of step 0 are zeros.
  const int rows = m.k == 1 ? N + 1 + 2 * F : N + 1;
  auto slot = [&](int s) { return ckpt + static_cast<size_t>(s / m.k) * rows * b.P; };
  if (ckpt)
    for (int r = 0; r < N; ++r) b.row(slot(0), r).store(0.0f);
  auto load = [&](int r) { return X.get(r); };
  float zn[F];
  load_z<F>(m, b, 0, zn);
  Ahead<F, U> ahead;
  pc_fetch<F, U>(ahead, m, 0, ctab, load);
  for (int s = 0; s < N; ++s) {
    float z[F], y[F], d[F];
#pragma unroll
    for (int f = 0; f < F; ++f) z[f] = zn[f];
    load_z<F>(m, b, min(s + 1, N - 1), zn);
    float xs;
    if (ckpt && s + 1 < N && (s + 1) % m.k == 0) {
      const float* next = slot(s + 1);
      xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load, [&](int r, float x) {
        X.set(r, x);
        b.row(next, r).store(x);
      });
    } else {
      xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load,
                      [&](int r, float x) { X.set(r, x); });
    }
    if (s + 1 < N) pc_fetch<F, U>(ahead, m, s + 1, ctab, load);
    if (ckpt && s % m.k == 0) {
      const float* c = slot(s) + static_cast<size_t>(N) * b.P;
      b.row(c).store(invB);
      if (m.k == 1) store_sums<F>(b, c + b.P, y, d);
    }
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
  // (the states are done with: their rows hold the wavefronts' sums)
  block_sum_to(static_cast<int>(threadIdx.x) < b.n ? static_cast<double>(v) : 0.0,
               reinterpret_cast<double*>(lds), part + blockIdx.x);
}

// ----------------------------------------------------------------------
// Backward.  scratch slot j (j < k) holds rows [0,N): start states of step
// s0+j, row N: 1/B at that step, rows N+1..N+2F: final sums y, d of step
// s0+j.  Slot 0's state rows are not used (the checkpoint is read instead).
// The step table is the forward's, read with scalar loads.  LDS: state
// adjoints [N][lanes], 40 960 bytes at 40 rates and 256 lanes: four blocks per
// CU; the block sums reuse its rows.
// ----------------------------------------------------------------------
template <int F, int BD, int U>
__global__ void __launch_bounds__(BD)
    k_price_bwd(KOO_MODEL_PARAMS, const float* __restrict__ vols, const float* __restrict__ ckpt,
                const float* __restrict__ tab, float* __restrict__ scratch,
                double* __restrict__ part) {
  KOO_MODEL_LOCAL;
  extern __shared__ float lds[];
  const BlockPaths b(m.P, blockIdx.x, BD);
  const int N = m.N;
  const c_cfloat ctab = cmem(tab);
  const LaneRows<BD> lam{lds + threadIdx.x};
  VegaSums<kVegaTiles<BD>> vegas;
  vegas.clear();
  for (int r = 0; r < N; ++r) lam.set(r, 0.0f);

  const size_t slot = static_cast<size_t>(N + 1 + 2 * F) * b.P;
  const int nseg = (N + m.k - 1) / m.k;
  float tail = 0.0f;
  Ahead<F, U> ahead;
  for (int seg = nseg - 1; seg >= 0; --seg) {
    const int s0 = seg * m.k;
    const int s1 = min(N, s0 + m.k);
    const bool every = m.k == 1;  // checkpoint holds the sums: no recompute
    const float* ck = ckpt + static_cast<size_t>(seg) * (every ? slot : (N + 1) * b.P);
    // Recompute the segment: state (and 1/B) at the start of step s0+j+1
    // into slot j+1 (the last step's is not needed), final sums of step s0+j
    // into slot j.
    for (int s = s0; s < (every ? s0 : s1); ++s) {
      const int j = s - s0;
      const float* src = j == 0 ? ck : scratch + j * slot;
      float* cur = scratch + j * slot;
      float* dst = cur + slot;
      const bool keep = s + 1 < s1;
      float z[F], y[F], d[F];
      load_z<F>(m, b, s, z);
      auto load = [&](int r) { return b.row(src, r).load(); };
      if (j == 0) pc_fetch<F, U>(ahead, m, s, ctab, load);
      const float xs = pc_step<F, U>(m, s, ctab, ahead, z, y, d, load, [&](int r, float x) {
        b.row(dst, r, keep).store(x);
      });
      if (keep)
        pc_fetch<F, U>(ahead, m, s + 1, ctab, [&](int r) { return b.row(dst, r).load(); });
      store_sums<F>(b, cur + static_cast<size_t>(N + 1) * b.P, y, d);
      if (keep) {
        const float fs = fmaf(start_level(m, s), fast_exp2(xs), -m.disp[s]);
        b.row(dst, N).store(b.row(src, N).load() * fast_rcp(1.0f + m.taus[s] * fs));
      }
    }
    // Reverse the segment's steps.
    for (int s = s1 - 1; s >= s0; --s) {
      const int j = s - s0;
      const float* src = j == 0 ? ck : scratch + j * slot;
      const float* sums = every ? ck : scratch + j * slot;
      auto load = [&](int r) { return b.row(src, r).load(); };
      reverse_fetch<F, U>(ahead, m, s, ctab, load, lam);
      const float invBs = b.row(src, N).load();
      float y[F], d[F];
      load_sums<F>(b, sums + static_cast<size_t>(N + 1) * b.P, y, d);
      reverse_step<F, U>(
          m, s, ctab, ahead, load, lam, y, d,
          [&](float& lp, float x) {
            // The rate fixing at the end of this step: caplet value and the
            // numeraire it enters for later fixings.  (Lanes past the last
            // path read 1/B = 0, so their adjoints stay zero.)
            const float tau = m.taus[s];
            const float xs = start_level(m, s) * fast_exp2(x);
            const float fs = xs - m.disp[s];
            const float inv = fast_rcp(1.0f + tau * fs);
            const float v = caplet_value(fs, tau, m.strike, inv);
            const float dv = caplet_deriv(fs, tau, m.strike, inv);
            lp = fmaf(dv * invBs - tau * inv * tail, kLn2 * xs, lp);
            tail += v * invBs;
          },
          vegas);
    }
  }
  adjoint_sums<BD>(m, vols, lds, vegas, part + static_cast<size_t>(blockIdx.x) * 2 * N);
}

// Blocks of 256 lanes, and of one wavefront for long curves, whose rows fill
// the LDS in smaller pieces, for few paths, which then reach more CUs, and for
// the shortest curves.
int block_lanes(int paths, int N) {
  return N >= kShortCurve && N <= 45 && paths >= 65536 ? 256 : 64;
}
size_t rows_lds(int N, int lanes) { return sizeof(float) * static_cast<size_t>(N) * lanes; }
// Floats of the checkpoint buffer before the step table.
size_t ckpt_floats(int paths, int N, int F, int k) {
  const size_t rows = k == 1 ? N + 1 + 2 * F : N + 1;
  return static_cast<size_t>((N + k - 1) / k) * rows * paths;
}
// Doubles of the partials before the step table of a forward without
// checkpoints.
size_t partial_doubles(int paths, int N) {
  const int t = block_lanes(paths, N);
  return (static_cast<size_t>(paths) + t - 1) / t * 2 * N;
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
        sizeof(float) * (ckpt_floats(paths, rates, factors, k) + step_table_floats(rates));
  // k == 1 needs no recompute scratch; one float keeps the pointer non-null.
  if (scratch_bytes)
    *scratch_bytes = k == 1 ? sizeof(float)
                            : sizeof(float) * static_cast<size_t>(k < rates ? k : rates) *
                                  (rates + 1 + 2 * factors) * P;
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
  Model m{variates, cmem(initial_rates), cmem(taus), cmem(displacements), cmem(pseudo_roots),
          strike, paths, rates,
          checkpoint_every};
  const int threads = block_lanes(paths, rates);
  const int blocks = (paths + threads - 1) / threads;
  const size_t lds = rows_lds(rates, threads);
  float* tab = checkpoints
                   ? checkpoints + ckpt_floats(paths, rates, factors, checkpoint_every)
                   : reinterpret_cast<float*>(partials + partial_doubles(paths, rates));
  hipStream_t st = as_stream(stream);
  switch (factors) {
#define KOO_FWD(F, BD, U)                                                                        \
  hipLaunchKernelGGL((k_price_fwd<F, BD, U>), dim3(blocks), dim3(BD), lds, st, m.z, m.f0,        \
                     m.taus, m.disp, m.A, m.strike, m.P, m.N, m.k, tab, checkpoints, partials)
#define KOO_CASE(F)                                                                              \
  case F:                                                                                        \
    hipLaunchKernelGGL(k_step_table<F>, dim3((rates * rates + 255) / 256), dim3(256), 0, st,     \
                       m.z, m.f0, m.taus, m.disp, m.A, m.strike, m.P, m.N, m.k, tab);            \
    if (threads == 256)                                                                          \
      KOO_FWD(F, 256, kWindow<F>);                                                               \
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
  hipLaunchKernelGGL(k_finalize_cols, dim3(1), dim3(256), 0, st, partials, blocks, 1,
                     1.0 / static_cast<double>(paths), price_out);
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
  Model m{variates, cmem(initial_rates), cmem(taus), cmem(displacements), cmem(pseudo_roots),
          strike, paths, rates,
          checkpoint_every};
  const int threads = block_lanes(paths, rates);
  const int blocks = (paths + threads - 1) / threads;
  const size_t lds = rows_lds(rates, threads);
  const float* tab = checkpoints + ckpt_floats(paths, rates, factors, checkpoint_every);
  hipStream_t st = as_stream(stream);
  switch (factors) {
#define KOO_BWD(F, BD, U)                                                                        \
  hipLaunchKernelGGL((k_price_bwd<F, BD, U>), dim3(blocks), dim3(BD), lds, st, m.z, m.f0,        \
                     m.taus, m.disp, m.A, m.strike, m.P, m.N, m.k, vols, checkpoints, tab,       \
                     segment_scratch, partials)
#define KOO_CASE(F)                                                                              \
  case F:                                                                                        \
    if (threads == 256)                                                                          \
      KOO_BWD(F, 256, kWindow<F>);                                                               \
    else if (rates >= kShortCurve)                                                               \
      KOO_BWD(F, 64, kWindow<F>);                                                                \
    else                                                                                         \
      KOO_BWD(F, 64, 1);                                                                         \
    break;
    KOO_CASE(1) KOO_CASE(2) KOO_CASE(3) KOO_CASE(4) KOO_CASE(5) KOO_CASE(6) KOO_CASE(7)
    KOO_CASE(8)
#undef KOO_CASE
#undef KOO_BWD
  }
  hipLaunchKernelGGL(k_finalize_cols, dim3(2 * rates), dim3(256), 0, st, partials, blocks,
                     2 * rates, 1.0 / static_cast<double>(paths), greeks_out);
  return check_launch("lmm_price_bwd");
}
