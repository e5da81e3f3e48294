// lmm_step.h -- device building blocks shared by the fused LMM kernels
// (caplet price/adjoint and the Bermudan swaption paths): wavefront and block
// reductions, the model arguments, and the predictor-corrector log-Euler step
// of LMM_evolver_all.cu:571-742 (spot measure, displaced diffusion).
#pragma once

#include <type_traits>

#include "koo_common.h"

namespace koo {
namespace lmm {
// Internal linkage: every kernel source gets its own copy.
namespace {

constexpr int kMaxRates = 90;
constexpr int kMaxFactors = 8;

__device__ __forceinline__ float fast_exp(float x) { return __expf(x); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// State of a rate: x = log2((f + d) / (f0 + d)).  Relative to its start the
// state is of the size of the path's own moves, so FP32 rounds it by 6e-8 of
// those and not of log f (about 3), and in base 2 the hardware exponential
// takes it as it is.  f + d = (f0 + d) 2^x.
constexpr float kLn2 = 0.693147180559945309417f;
constexpr float kLog2e = 1.442695040888963407360f;
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Drift coefficient in the state's units, G = log2(e) g with
// g = tau (f + d) / (1 + tau f), from the state: g = 1 / (1 + (1/tau - d) /
// (f + d)), so G = 1 / (ln2 + kr 2^-x) with kr = ln2 (1/tau - d) / (f0 + d)
// (one multiply-add between the two hardware transcendentals).
__device__ __forceinline__ float drift_coeff(float x, float kr) {
  return fast_rcp(fmaf(kr, fast_exp2(-x), kLn2));
}
// dG/dx = g (1 - g) = G drift_slope(G)
__device__ __forceinline__ float drift_slope(float G) { return fmaf(G, -kLn2 * kLn2, kLn2); }

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Agent-scope (device-wide) coherent store and load of a double: the store
// writes through the XCD's L2, the load misses it, so values exchanged
// between blocks of one running kernel need no cache write-back or
// invalidation (used by the persistent kernels for their block partials).
__device__ __forceinline__ void store_agent(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double load_agent(const double* p) {
  return __hip_atomic_load(const_cast<double*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Block-wide FP64 sum of one value per lane into part[col]; every lane of the
// block must call it (contains barriers).  Agent: the store is agent-coherent.
template <bool Agent = false>
__device__ __forceinline__ void block_sum_to(double v, double* scratch_lds, double* out) {
  v = wave_sum_f64(v);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch_lds[w] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int i = 0; i < static_cast<int>(blockDim.x >> 6); ++i) t += scratch_lds[i];
    if (Agent)
      store_agent(out, t);
    else
      *out = t;
  }
}

// Constant address space (4): the model's curve and pseudo-roots are read
// through it, since no kernel writes them, so that their uniform reads use
// the scalar cache also where the model comes from a device descriptor (the
// batched and persistent kernels), not only from __restrict__ arguments.
#if defined(__HIP_DEVICE_COMPILE__)
#define KOO_CONSTANT __attribute__((address_space(4)))
#else
#define KOO_CONSTANT
#endif
typedef const float KOO_CONSTANT* c_cfloat;
template <class P>
__host__ __device__ __forceinline__ c_cfloat cmem(P p) {
  return (c_cfloat)p;
}

struct Model {
  const float* z;     // (S,F,P) bridged variates
  c_cfloat f0;        // N
  c_cfloat taus;      // N
  c_cfloat disp;      // N
  c_cfloat A;         // (S,N,F)
  float strike;
  int P, N;
  int S1, L;  // SweepPlan of the adjoint
};

// What the forward keeps for the reverse sweep, in the rows (of P) that the
// checkpoint interval pays for.  The reverse of a step needs that step's final
// sums and the states after it: it recovers the states before it from them
// (reverse_step), so no step's states have to be kept but the last's.  Steps
// 0..S1-1 keep their sums (2F rows each); as many as the checkpoint buffer
// holds.  The later steps are run again in segments of L, whose sums the
// segment scratch holds, from the states at S1, S1 + L, ...
// Checkpoint rows: the sums; the N states when step S1 begins (those of rates
// that have fixed as they fixed) and 1/B there; then per further segment the
// alive states and 1/B when it begins.  1/B takes two rows (Deflator); where it
// has not moved out of FP32's range yet, at step 0 and on a single rate, one.
struct SweepPlan {
  int S1, L;
};
__host__ __device__ constexpr int sweep_state_row(int F, int S1) { return 2 * F * S1; }
__host__ __device__ constexpr bool sweep_exponent_row(int N, int S1) { return S1 > 0 && N > 1; }
// Rows up to and including segment 0's.
__host__ __device__ constexpr int sweep_first_rows(int N, int F, int S1) {
  return 2 * F * S1 + N + 1 + (sweep_exponent_row(N, S1) ? 1 : 0);
}
// First row of segment i >= 1, which begins at step S1 + i L.
__host__ __device__ constexpr int sweep_segment_row(int N, int F, int S1, int L, int i) {
  return sweep_first_rows(N, F, S1) + (i - 1) * (N - S1 + 2) - L * (i * (i - 1) / 2);
}
// Rows of the checkpoint buffer and of the segment scratch at interval k.
inline int ckpt_rows(int N, int F, int k) {
  return k == 1 ? N * (N + 1 + 2 * F) : (N + k - 1) / k * (N + 1);
}
inline int scratch_rows(int N, int F, int k) {
  return k == 1 ? 0 : (k < N ? k : N) * (N + 1 + 2 * F);
}
// (With S1 = 0 the segments are at least k long, and each takes at most N + 1
// rows: a plan always exists.)
inline SweepPlan sweep_plan(int N, int F, int k) {
  if (k == 1) return {N, N};
  const int room = ckpt_rows(N, F, k);
  int L = scratch_rows(N, F, k) / (2 * F);
  if (L > N) L = N;
  int S1 = N;
  for (; S1 > 0; --S1) {
    const int more = (N - S1 + L - 1) / L;  // segments
    const int rows =
        more > 1 ? sweep_segment_row(N, F, S1, L, more) : sweep_first_rows(N, F, S1);
    if (rows <= room) break;
  }
  return {S1, L};
}

// 1/B of a path as m 2^e, m in [0.5, 1): on a path whose rates run away it falls
// below FP32's range while the caplets that paid before still count, and the
// reverse, which multiplies it back step by step, has to come out at theirs.
struct Deflator {
  float m = 1.0f;
  int e = 0;
  __device__ __forceinline__ void scale(float by) {
    m *= by;
    e += __builtin_amdgcn_frexp_expf(m);
    m = __builtin_amdgcn_frexp_mantf(m);
  }
  __device__ __forceinline__ float value() const { return ldexpf(m, e); }
};

// The step table: for every step s and alive rate r >= s the pair
// {fixed drift c = -0.5 log2(e) sum_f A(s,r,f)^2, kr of drift_coeff}, steps one
// after the other (N - s pairs each): N (N + 1) floats.
__host__ __device__ constexpr size_t step_table_floats(int N) {
  return static_cast<size_t>(N) * N + N;
}
// First float of step s.
__host__ __device__ constexpr int step_table_row(int N, int s) { return s * (2 * N + 1 - s); }

// A rate's f + d at the start, by which 2^x is scaled.
__device__ __forceinline__ float start_level(const Model& m, int r) { return m.f0[r] + m.disp[r]; }

// kr of drift_coeff; NaN below zero, where a rate has no logarithm: NaN is then
// what the rate, those above it and the price come to.
__device__ __forceinline__ float drift_constant(const Model& m, int r) {
  const float level = start_level(m, r);
  return level < 0.0f ? __builtin_nanf("") : kLn2 * (1.0f / m.taus[r] - m.disp[r]) / level;
}

// Entry q < N * N of the square (s, r) = (q / N, q % N) into the table (nothing
// below the diagonal).  One function for every copy of the table, so an LDS
// copy and a global one hold the same bits.
template <int F>
__device__ __forceinline__ void put_step_entry(const Model& m, int q, float* tab) {
  const int s = q / m.N, r = q - s * m.N;
  if (r < s) return;
  c_cfloat a = m.A + static_cast<size_t>(q) * F;
  float c = 0.0f;
#pragma unroll
  for (int f = 0; f < F; ++f) c = fmaf(a[f], a[f], c);
  float* t = tab + step_table_row(m.N, s) + 2 * (r - s);
  t[0] = -0.5f * kLog2e * c;
  t[1] = drift_constant(m, r);
}

// Every lane of the block takes part; the caller then synchronises.
template <int F>
__device__ __forceinline__ void fill_step_table(const Model& m, float* tab) {
  for (int q = threadIdx.x; q < m.N * m.N; q += blockDim.x) put_step_entry<F>(m, q, tab);
}

// One value per lane and rate in LDS: lane-minor rows of BD lanes, so a
// wavefront's access is free of bank conflicts and, BD being a constant, the
// rows of a window are offsets of one address.
template <int BD>
struct LaneRows {
  float* p;  // this lane's column
  __device__ __forceinline__ float get(int r) const { return p[r * BD]; }
  __device__ __forceinline__ void set(int r, float v) const { p[r * BD] = v; }
};

// A block's part of one row of a path-minor array in global memory, as a
// buffer: lanes past the last path read zero and store nothing (the buffer's
// range check), and the row's address stays in scalar registers, so an access
// costs no vector instruction but itself (a 64-bit pointer per lane costs an
// add with carry each time).
struct PathRow {
  __amdgpu_buffer_rsrc_t r;
  int byte;
  __device__ __forceinline__ float load() const {
    return __int_as_float(static_cast<int>(__builtin_amdgcn_raw_buffer_load_b32(r, byte, 0, 0)));
  }
  __device__ __forceinline__ void store(float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(static_cast<unsigned>(__float_as_int(v)), r, byte, 0, 0);
  }
};

// The paths of a block: paths p0 .. p0 + n - 1 (n at most the lanes), one lane
// each.
struct BlockPaths {
  size_t p0, P;
  int n;
  __device__ __forceinline__ BlockPaths(int paths, int block, int lanes)
      : p0(static_cast<size_t>(block) * lanes), P(paths), n(min(lanes, static_cast<int>(P - p0))) {}
  // `base`: element 0 of the row
  __device__ __forceinline__ PathRow row(const float* base) const {
    return PathRow{
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base) + p0, 0, 4 * n, 0x00027000),
        static_cast<int>(4 * threadIdx.x)};
  }
  // P, out of the compiler's sight: rows addressed with it inside a loop are
  // formed there, where many of them would be hoisted out of it into more
  // scalar registers than there are
  __device__ __forceinline__ size_t stride() const {
    size_t q = P;
    asm volatile("" : "+s"(q));
    return q;
  }
  // row `r` of an array of rows of P
  __device__ __forceinline__ PathRow row(const float* base, int r) const {
    return row(base + static_cast<size_t>(r) * P);
  }
};

// The same in global memory (rows of P), for blocks whose LDS has no room.
struct GlobalRows {
  BlockPaths b;
  float* rows;
  __device__ __forceinline__ float get(int r) const { return b.row(rows, r).load(); }
  __device__ __forceinline__ void set(int r, float v) const { b.row(rows, r).store(v); }
};

// Vega terms of a wavefront, summed over its lanes on the matrix cores: the
// term of the rate j places from the top is the A operand of a 16x16x4 product
// whose B is one in column j mod 16, so column j of tile j / 16 collects 16
// partial sums (of four lanes each) over all steps.  Two issue slots a rate
// (the one-hot column and the product), where folding the 64 lanes by DPP and
// adding to LDS takes about eight.  The terms have to be finite (zero times
// infinity would reach the other columns): see NonFinite.
template <int TILES>
struct VegaSums {
  typedef float f4 __attribute__((ext_vector_type(4)));
  f4 acc[TILES];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int t = 0; t < TILES; ++t) acc[t] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  // terms of the rates j0 .. j0 + U - 1 from the top, all of one tile
  template <int U>
  __device__ __forceinline__ void add(int j0, const float (&w)[U]) {
    const unsigned long long col = 0x0001000100010001ull << (j0 & 15);
    float one[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      one[u] = __builtin_amdgcn_inverse_ballot_w64(col << u) ? 1.0f : 0.0f;
#pragma unroll
    for (int t = 0; t < TILES; ++t)
      if ((j0 >> 4) == t) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u], one[u], acc[t], 0, 0, 0);
      }
  }
  // put(j, v): the wavefront's sum of the rate j places from the top, one lane
  // per rate
  template <class Put>
  __device__ __forceinline__ void sums(int rates, Put put) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      double v = (static_cast<double>(acc[t][0]) + static_cast<double>(acc[t][1])) +
                 (static_cast<double>(acc[t][2]) + static_cast<double>(acc[t][3]));
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (lane < 16 && 16 * t + lane < rates) put(16 * t + lane, v);
    }
  }
};

// A path's adjoints that are infinite or NaN.  States and what the reverse forms
// from them are finite; an adjoint becomes infinite or NaN only where it begins,
// at a fixing or a payoff whose rate has left FP32's range, and from there
// reaches the rates below.  There it is set to zero and its rate remembered, and
// the Greeks of that rate and those below are made NaN in the end: the rates
// above keep theirs.  (Caught at each term instead, the caplet backward took 5%
// longer.)
struct NonFinite {
  int rate = -1;  // the highest of them
  __device__ __forceinline__ void take(float& lp, int r) {
    const bool finite = fabsf(lp) < __builtin_inff();
    lp = finite ? lp : 0.0f;
    rate = finite ? rate : max(rate, r);
  }
};

// The variates of step s.
template <int F>
__device__ __forceinline__ void load_z(const Model& m, const BlockPaths& b, int s, float (&z)[F]) {
  const size_t P = b.stride();
  const float* zs = m.z + static_cast<size_t>(s) * F * P;
#pragma unroll
  for (int f = 0; f < F; ++f, zs += P) z[f] = b.row(zs).load();
}

// A step's final sums y, d in the 2F rows at `rows`.
template <int F>
__device__ __forceinline__ void store_sums(const BlockPaths& b, const float* rows,
                                           const float (&y)[F], const float (&d)[F]) {
  const size_t P = b.stride();
#pragma unroll
  for (int f = 0; f < F; ++f, rows += P) b.row(rows).store(y[f]);
#pragma unroll
  for (int f = 0; f < F; ++f, rows += P) b.row(rows).store(d[f]);
}
template <int F>
__device__ __forceinline__ void load_sums(const BlockPaths& b, const float* rows, float (&y)[F],
                                          float (&d)[F]) {
  const size_t P = b.stride();
#pragma unroll
  for (int f = 0; f < F; ++f, rows += P) y[f] = b.row(rows).load();
#pragma unroll
  for (int f = 0; f < F; ++f, rows += P) d[f] = b.row(rows).load();
}

// Rates per window of the step loops: a window's uniform data (pseudo-roots,
// fixed drifts, drift constants) is contiguous and is fetched into scalar
// registers in a few wide loads while the window before it is worked on.
// Scalar loads return out of order, so any wait for one is a wait for all of
// them: one wait per window of four rates instead of one per load.  (A load at
// each use cost 215 ns a rate update where one wavefront has a SIMD: the
// caplet forward at 4096 paths, 40 rates and 5 factors took 179 us, 118 with
// the windows.)  Two buffers of four rates take 8 (F + 2) scalar registers, too
// many beyond six factors.
// Curves shorter than a window run windows of one rate (U = 1).
template <int F>
constexpr int kWindow = F <= 6 ? 4 : 2;
constexpr int kShortCurve = 4;  // rates below which U = 1

template <int F, int U>
struct Rows {
  float a[U][F], c[U], kr[U];
};

// Rows r0 .. r0 + U - 1 of step s, 0 <= r0 <= N - U.  Those below rate s are
// not the step's and are not used (for the pseudo-roots they are dead rates of
// the step; in the triangular table they belong to the step before: r0 < s
// only where s > N - U, so the index stays positive).
template <int F, int U, class Tab>
__device__ __forceinline__ void load_rows(Rows<F, U>& w, const Model& m, Tab tab, int s, int r0) {
  // 32-bit offset: keeps the address scalar
  c_cfloat A = m.A + (s * m.N + r0) * F;
  const auto t = tab + (step_table_row(m.N, s) + 2 * (r0 - s));
#pragma unroll
  for (int i = 0; i < U; ++i) {
#pragma unroll
    for (int f = 0; f < F; ++f) w.a[i][f] = A[i * F + f];
    w.c[i] = t[2 * i];
    w.kr[i] = t[2 * i + 1];
  }
}

// Waits for the scalar and LDS loads issued so far and keeps the compiler from
// moving later ones above: the loads that follow are then still in flight while
// the window is worked on.
__device__ __forceinline__ void window_ready() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_sched_barrier(0);
}

// Uniform values carried round a loop, held in scalar registers (the compiler
// would carry what only vector instructions use in vector registers).  `x` has
// to be what the compiler itself takes for uniform (read with uniform addresses
// and not spilled to a lane's register on the way): "+s" makes it an error where
// it is not, "illegal VGPR to SGPR copy", as when the library is compiled with
// packed FP32.  The remedy is a __builtin_amdgcn_readfirstlane on x.
__device__ __forceinline__ float keep_scalar(float x) {
  int i = __float_as_int(x);
  asm volatile("" : "+s"(i));
  return __int_as_float(i);
}
// (A table in LDS is read into vector registers and stays there.)
template <class Tab, int F, int U>
__device__ __forceinline__ void keep_scalar(Rows<F, U>& w) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int f = 0; f < F; ++f) w.a[u][f] = keep_scalar(w.a[u][f]);
    if constexpr (std::is_same<Tab, c_cfloat>::value) {
      w.c[u] = keep_scalar(w.c[u]);
      w.kr[u] = keep_scalar(w.kr[u]);
    }
  }
}

// Windows of the alive rates s..N-1.  Ascending, all but the first are full and
// the last ends at rate N - 1: the first holds rates s .. part_end - 1.
// Descending they start at rate N - 1 and the last holds rate s.  The window
// with rate s is read at part_base, where U rows of the step exist.
template <int U>
__device__ __forceinline__ int part_end(int N, int s) {
  return N - (N - s - 1) / U * U;
}
template <int U>
__device__ __forceinline__ int part_base(int N, int s) {
  return min(s, N - U);
}

// A fetched window.  The step loops work on two in turn (no copies: a copy of
// a register waits for the load into it), the first of a step fetched while
// the step before it ends.
template <int F, int U>
struct Ahead {
  Rows<F, U> rows;
  float x[U];  // states
  float l[U];  // the adjoints (the reverse)

  // Waits for the window, before the next one's loads are issued.
  template <class Tab>
  __device__ __forceinline__ void take() {
    window_ready();
    keep_scalar<Tab>(rows);
  }
};
// Between the loads of the next window and the work on this one.
__device__ __forceinline__ void loads_issued() { __builtin_amdgcn_sched_barrier(0); }

// Fetches the first window of PC step s; `load(r)` gives the state of rate r.
template <int F, int U, class Tab, class Load>
__device__ __forceinline__ void pc_fetch(Ahead<F, U>& h, const Model& m, int s, Tab tab,
                                         Load load) {
  const int base = part_base<U>(m.N, s);
  load_rows<F, U>(h.rows, m, tab, s, base);
#pragma unroll
  for (int i = 0; i < U; ++i) h.x[i] = load(base + i);
}

// One predictor-corrector step s over the alive rates.  In the state's units
//   G_r  = drift_coeff(x_r)          y_f += G_r a_rf  (y starts at log2(e) z)
//   xh_r = x_r + c_r + sum_f a_rf y_f
//   Gh_r = drift_coeff(xh_r)         d_f += (Gh_r - G_r) a_rf
//   x'_r = xh_r + 0.5 sum_f a_rf d_f
// which is the log-Euler step with drift mu = sum a e, e = sum G a, and the
// corrector's half difference of the drifts: y carries the diffusion along
// with the predictor drift, d the difference of the two drift sums, so a
// rate takes four F-term sums instead of five.  `h`: pc_fetch of this step.
// `load(r)` gives the state of rate r, `store(r, x)` takes its new one; y and d
// return the final sums, the function the new state of the fixing rate s.
template <int F, int U, class Tab, class Load, class Store>
__device__ __forceinline__ float pc_step(const Model& m, int s, Tab tab, Ahead<F, U>& h,
                                         const float (&z)[F], float (&y)[F], float (&d)[F],
                                         Load load, Store store) {
  const int N = m.N;
#pragma unroll
  for (int f = 0; f < F; ++f) {
    y[f] = kLog2e * z[f];
    d[f] = 0.0f;
  }
  auto rate = [&](const Rows<F, U>& w, int u, float x, int r) {
    const float G = drift_coeff(x, w.kr[u]);
    float xh = x + w.c[u];
#pragma unroll
    for (int f = 0; f < F; ++f) {
      y[f] = fmaf(G, w.a[u][f], y[f]);
      xh = fmaf(w.a[u][f], y[f], xh);
    }
    const float g = drift_coeff(xh, w.kr[u]) - G;
    float dd = 0.0f;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      d[f] = fmaf(g, w.a[u][f], d[f]);
      dd = fmaf(w.a[u][f], d[f], dd);
    }
    const float xn = fmaf(0.5f, dd, xh);
    store(r, xn);
    return xn;
  };
  Ahead<F, U> g;
  auto fetch = [&](Ahead<F, U>& to, int r) {
    load_rows<F, U>(to.rows, m, tab, s, r);
#pragma unroll
    for (int u = 0; u < U; ++u) to.x[u] = load(r + u);
  };
  auto window = [&](const Ahead<F, U>& w, int r0) {
    loads_issued();
#pragma unroll
    for (int u = 0; u < U; ++u) rate(w.rows, u, w.x[u], r0 + u);
  };
  const int base = part_base<U>(N, s), end = part_end<U>(N, s);
  float first = 0.0f;
  h.template take<Tab>();
  if (end < N) fetch(g, end);
  loads_issued();
#pragma unroll
  for (int i = 0; i < U; ++i)
    if (base + i >= s && base + i < end) {
      const float v = rate(h.rows, i, h.x[i], base + i);
      if (base + i == s) first = v;
    }
  int r0 = end;
  for (; r0 + U < N; r0 += 2 * U) {
    g.template take<Tab>();
    fetch(h, r0 + U);
    window(g, r0);
    h.template take<Tab>();
    if (r0 + 2 * U < N) fetch(g, r0 + 2 * U);
    window(h, r0 + U);
  }
  if (r0 < N) {
    g.template take<Tab>();
    window(g, r0);
  }
  return first;
}

// Fetches the first window of the reverse of step s (rates N-1, N-2, ...): a
// full one, or the one with rate s.
template <int F, int U, class Tab, class States, class Lanes>
__device__ __forceinline__ void reverse_fetch(Ahead<F, U>& h, const Model& m, int s, Tab tab,
                                              const States& X, const Lanes& lam) {
  load_rows<F, U>(h.rows, m, tab, s, m.N - U);
#pragma unroll
  for (int i = 0; i < U; ++i) {
    h.x[i] = X.get(m.N - U + i);
    h.l[i] = lam.get(m.N - U + i);
  }
}

// Reverse of PC step s over the rates N-1..s.  On entry `X` holds the states
// and `lam` their adjoints after the step, on exit those before it; y / d are
// the step's final sums.  With the sums after rate r (un-accumulated as the
// rates descend) the step runs backwards by itself,
//   xh_r = x'_r - 0.5 sum a d,   x_r = xh_r - c_r - sum a y,
// so the states before the step need not be kept.  (Each step back rounds
// the states once more, about as the step forward does.)  `h`: reverse_fetch
// of this step.  `fixing(lp, x')` adds the product's adjoint of the rate
// fixing at the end of the step (r == s) to lp; `vegas` takes
// w = sum_f Abar(s,r,f) A(s,r,f) of the step, which contracts to scalars the
// reverse already has: with the adjoint sums D of d and Y of y (rates
// descending),
//   D_f += 0.5 lp a_f, q = sum a D;   xhb = lp + q dGh/dx
//   Y_f += xhb a_f,    p = sum a Y;   lam = xhb + (p - q) dG/dx
//   w = 0.5 lp sum a d + Gh q + G (p - q) + xhb (sum a y + 2 c).
template <int F, int U, class Tab, class States, class Lanes, class Fixing, class Vegas>
__device__ __forceinline__ void reverse_step(const Model& m, int s, Tab tab, Ahead<F, U>& h,
                                             const States& X, const Lanes& lam, float (&y)[F],
                                             float (&d)[F], Fixing fixing, Vegas& vegas) {
  const int N = m.N;
  float D[F], Y[F];
#pragma unroll
  for (int f = 0; f < F; ++f) D[f] = Y[f] = 0.0f;
  auto rate = [&](const Rows<F, U>& v, int u, float xe, float lp, int r, bool may_fix) {
    const float c = v.c[u];
    float my = 0.0f, md = 0.0f;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      md = fmaf(v.a[u][f], d[f], md);
      my = fmaf(v.a[u][f], y[f], my);
    }
    const float xh = fmaf(-0.5f, md, xe);
    const float mc = my + c;
    const float x = xh - mc;
    const float Gh = drift_coeff(xh, v.kr[u]);
    const float G = drift_coeff(x, v.kr[u]);
    X.set(r, x);
    if (may_fix && r == s) fixing(lp, xe);
    const float lh = 0.5f * lp;
    float q = 0.0f;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      D[f] = fmaf(lh, v.a[u][f], D[f]);
      q = fmaf(v.a[u][f], D[f], q);
    }
    const float uh = Gh * q;
    const float xhb = fmaf(uh, drift_slope(Gh), lp);
    float p = 0.0f;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      Y[f] = fmaf(xhb, v.a[u][f], Y[f]);
      p = fmaf(v.a[u][f], Y[f], p);
    }
    const float ug = G * (p - q);
    lam.set(r, fmaf(ug, drift_slope(G), xhb));
    const float g = Gh - G;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      y[f] = fmaf(-G, v.a[u][f], y[f]);
      d[f] = fmaf(-g, v.a[u][f], d[f]);
    }
    // uh + ug, as one multiply-add written out: left to the compiler, the single,
    // batched and persistent kernels would not all round it alike
    return fmaf(xhb, mc + c, fmaf(lh, md, fmaf(G, p - q, uh)));
  };
  Ahead<F, U> g;
  auto fetch = [&](Ahead<F, U>& to, int r) {
    load_rows<F, U>(to.rows, m, tab, s, r);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      to.x[i] = X.get(r + i);
      to.l[i] = lam.get(r + i);
    }
  };
  auto window = [&](const Ahead<F, U>& v, int r0) {
    loads_issued();
    float w[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      w[u] = rate(v.rows, U - 1 - u, v.x[U - 1 - u], v.l[U - 1 - u], r0 + U - 1 - u, false);
    vegas.add(N - U - r0, w);
  };
  // full windows [r0, r0 + U); the window after the last of them is at base
  const int base = part_base<U>(N, s), end = part_end<U>(N, s);
  int r0 = N - U;
  for (; r0 - U >= end; r0 -= 2 * U) {
    h.template take<Tab>();
    fetch(g, r0 - U);
    window(h, r0);
    g.template take<Tab>();
    fetch(h, r0 - 2 * U >= end ? r0 - 2 * U : base);
    window(g, r0 - U);
  }
  if (r0 >= end) {
    h.template take<Tab>();
    fetch(g, base);
    window(h, r0);
    h = g;
  }
  // the window with rate s
  h.template take<Tab>();
  loads_issued();
#pragma unroll
  for (int i = U - 1; i >= 0; --i)
    if (base + i >= s && base + i < end) {
      const float w[1] = {rate(h.rows, i, h.x[i], h.l[i], base + i, true)};
      vegas.add(N - 1 - base - i, w);
    }
}

// Reverses the steps hi - 1 .. lo, whose sums are the 2F rows per step from
// `sums` (step lo's first), fetched a step ahead.
template <int F, int U, class Tab, class States, class Lanes, class Before, class Fixing,
          class Vegas>
__device__ __forceinline__ void reverse_steps(const Model& m, const BlockPaths& b, int hi, int lo,
                                              const float* sums, Tab tab, const States& X,
                                              const Lanes& lam, Before before, Fixing fixing,
                                              Vegas& vegas) {
  if (hi <= lo) return;
  const size_t step_rows = 2 * F * b.P;
  float yn[F], dn[F];
  load_sums<F>(b, sums + (hi - 1 - lo) * step_rows, yn, dn);
  Ahead<F, U> ahead;
  for (int s = hi - 1; s >= lo; --s) {
    before(s);
    reverse_fetch<F, U>(ahead, m, s, tab, X, lam);
    float y[F], d[F];
#pragma unroll
    for (int f = 0; f < F; ++f) {
      y[f] = yn[f];
      d[f] = dn[f];
    }
    if (s > lo) load_sums<F>(b, sums + (s - 1 - lo) * step_rows, yn, dn);
    reverse_step<F, U>(m, s, tab, ahead, X, lam, y, d,
                       [&](float& lp, float x) { fixing(s, lp, x); }, vegas);
  }
}

// Copies rows [lo, hi) of the states to or from the rows at `rows`.
template <class Lanes>
__device__ __forceinline__ void dump_states(const BlockPaths& b, const Lanes& X, const float* rows,
                                            int lo, int hi) {
#pragma unroll 4
  for (int r = lo; r < hi; ++r) b.row(rows, r - lo).store(X.get(r));
}
template <class Lanes>
__device__ __forceinline__ void load_states(const BlockPaths& b, const Lanes& X, const float* rows,
                                            int lo, int hi) {
#pragma unroll 4
  for (int r = lo; r < hi; ++r) X.set(r, b.row(rows, r - lo).load());
}

// Walks the alive rates s..N-1 of a curve, upwards or downwards, in windows
// whose uniform data is fetched a window ahead (as pc_step's):
// step(r, f + d, f, tau) with f + d = start_level 2^x.
template <int U, bool Down, class Lanes, class Step>
__device__ __forceinline__ void walk_curve(const Model& m, int s, const Lanes& X, Step step) {
  const int N = m.N;
  float f0n[U], dn[U], tn[U], xn[U], f0[U], d[U], tau[U], x[U];
  auto fetch = [&](int r) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      f0n[i] = m.f0[r + i];
      dn[i] = m.disp[r + i];
      tn[i] = m.taus[r + i];
      xn[i] = X.get(r + i);
    }
  };
  auto take = [&](bool more, int r) {
    window_ready();
#pragma unroll
    for (int i = 0; i < U; ++i) {
      f0[i] = keep_scalar(f0n[i]);
      d[i] = keep_scalar(dn[i]);
      tau[i] = keep_scalar(tn[i]);
      x[i] = xn[i];
    }
    if (more) fetch(r);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto one = [&](int i, int r) {
    const float v = (f0[i] + d[i]) * fast_exp2(x[i]);
    step(r, v, v - d[i], tau[i]);
  };
  const int base = part_base<U>(N, s), end = part_end<U>(N, s);
  if (!Down) {
    fetch(base);
    take(end < N, end);
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (base + i >= s && base + i < end) one(i, base + i);
    for (int r0 = end; r0 < N; r0 += U) {
      take(r0 + U < N, r0 + U);
#pragma unroll
      for (int i = 0; i < U; ++i) one(i, r0 + i);
    }
  } else {
    fetch(end < N ? N - U : base);
    for (int r0 = N - U; r0 >= end; r0 -= U) {
      take(true, r0 - U >= end ? r0 - U : base);
#pragma unroll
      for (int i = U - 1; i >= 0; --i) one(i, r0 + i);
    }
    take(false, 0);
#pragma unroll
    for (int i = U - 1; i >= 0; --i)
      if (base + i >= s && base + i < end) one(i, base + i);
  }
}

// Lanes of the adjoint's blocks.  Four wavefronts: a CU spreads those over its
// four SIMDs, where blocks of one or two that fill its LDS are left uneven (at
// 2^20 paths and 40 rates, 128-lane blocks took 2.93 ms in the backward, 256
// lanes 2.37, with the same eight wavefronts per CU).  One wavefront for few
// paths and for curves whose rows leave no room for two such blocks.
constexpr int kAdjLanes = 256, kAdjRates = 40;
// Rates that the batched and persistent kernels take.
constexpr int kBatchRates = 45;
template <int BD>
constexpr int kVegaTiles = (BD == kAdjLanes ? kBatchRates + 15 : kMaxRates + 15) / 16;

// Wavefronts of `paths` paths, and this one's index: every wavefront writes its
// own partial sums (so they do not depend on the block size), column after
// column: column c of wavefront w at part[c * waves + w].
__host__ __device__ constexpr int wave_count(int paths) { return (paths + 63) >> 6; }
template <int BD>
__device__ __forceinline__ int wave_index(int block) {
  return block * (BD / 64) + static_cast<int>(threadIdx.x >> 6);
}
template <bool Agent>
__device__ __forceinline__ void put_partial(double* part, int waves, int w, int col, double v) {
  double* o = part + static_cast<size_t>(col) * waves + w;
  if (w >= waves) return;
  if (Agent) store_agent(o, v);
  else *o = v;
}

// A wavefront's sums of the state adjoints and vega terms, as deltas
// (d/df0_r = log2(e) lam_r / (f0_r + d_r)) and vegas (over sigma_r): columns
// 0..N-1 and N..2N-1, NaN where `bad` says so.  Agent: the stores are
// agent-coherent.
template <int BD, bool Agent = false, class Lanes, class Vegas>
__device__ __forceinline__ void adjoint_sums(const Model& m, const float* __restrict__ vols,
                                             const Lanes& lam, const Vegas& vegas,
                                             const NonFinite& bad, double* part, int block) {
  const int N = m.N, lane = threadIdx.x & 63;
  int nan_to = bad.rate;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) nan_to = max(nan_to, __shfl_xor(nan_to, o, 64));
  const auto at = [&](int r, double v) { return r <= nan_to ? __builtin_nan("") : v; };
  const int waves = wave_count(m.P), w = wave_index<BD>(block);
  // four rates at a time, so that their butterflies overlap
  for (int r0 = 0; r0 < N; r0 += 4) {
    double v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = static_cast<double>(lam.get(min(r0 + i, N - 1)));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += __shfl_xor(v[i], o, 64);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (lane == i && r0 + i < N)
        put_partial<Agent>(part, waves, w, r0 + i,
                           at(r0 + i, v[i] * static_cast<double>(kLog2e) /
                                          static_cast<double>(start_level(m, r0 + i))));
  }
  vegas.sums(N, [&](int j, double v) {
    const int r = N - 1 - j;
    put_partial<Agent>(part, waves, w, N + r, at(r, v / static_cast<double>(vols[r])));
  });
}

// The model arrays are separate __restrict__ kernel arguments (not members of
// a by-value struct) so the compiler may read them through the scalar cache.
#define KOO_MODEL_PARAMS                                                                  \
  const float* __restrict__ z_, const float* __restrict__ f0_,                            \
      const float* __restrict__ taus_, const float* __restrict__ disp_,                   \
      const float* __restrict__ A_, float strike_, int P_, int N_, int S1_, int L_
#define KOO_MODEL_LOCAL \
  const Model m{z_, cmem(f0_), cmem(taus_), cmem(disp_), cmem(A_), strike_, P_, N_, S1_, L_}

// Batched kernels read the pointers of their device descriptor tables as
// global-memory pointers (address space 1), so accesses through them are
// global, not flat, instructions (flat ones also count against the LDS wait
// counter, which would serialise the state prefetch against the LDS
// traffic).  The host fills the same layout with plain pointers.
#if defined(__HIP_DEVICE_COMPILE__)
#define KOO_GLOBAL __attribute__((address_space(1)))
#else
#define KOO_GLOBAL
#endif
typedef const float KOO_GLOBAL g_cfloat;
typedef const double KOO_GLOBAL g_cdouble;
typedef float KOO_GLOBAL g_float;
typedef double KOO_GLOBAL g_double;
typedef int KOO_GLOBAL g_int;
// Address space 1 -> generic (the compiler keeps track that it is global).
template <class T>
__device__ __forceinline__ T* gmem(T KOO_GLOBAL* p) {
  return (T*)p;
}

// Batched launches number their blocks item after item; the item owning
// `block` is the last one whose first block (the member `first`) is <= block
// (binary search, uniform per block).
template <class Item>
__device__ __forceinline__ int find_block_owner(const Item* items, int n, int block,
                                                int Item::*first) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (items[mid].*first <= block) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Rate-count class of a product in the batched LS launches (a launch per class,
// so LDS is reserved for the class's largest curve).
inline int rate_class(int rates) {
  return rates <= 16 ? 0 : (rates <= 24 ? 1 : (rates <= 32 ? 2 : 3));
}

// out[col] = (sum_b part[b*ncols + col]) * scale, compensated; called by a
// whole block (k_finalize_cols runs one block per column).  Agent: the
// partials are read with agent-coherent loads.
template <bool Agent = false>
__device__ __forceinline__ void finalize_col(const double* __restrict__ part, int nb, int ncols,
                                             int col, double scale, double* __restrict__ out) {
  __shared__ double sv[16], sc[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  // per lane: Neumaier over a strided slice of the blocks
  // (eight loads in flight: one at a time took 30 us for 2^14 blocks)
  double s = 0.0, c = 0.0;
  for (int b0 = threadIdx.x; b0 < nb; b0 += 8 * blockDim.x) {
    double v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int b = b0 + i * static_cast<int>(blockDim.x);
      const double* src = part + static_cast<size_t>(b < nb ? b : 0) * ncols + col;
      const double x = Agent ? load_agent(src) : *src;
      v[i] = b < nb ? x : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const double x = v[i], t = s + x;
      c += (fabs(s) >= fabs(x)) ? (s - t) + x : (x - t) + s;
      s = t;
    }
  }
  // wavefront butterfly with error-free additions (TwoSum), then the waves
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double s2 = __shfl_xor(s, o, 64), c2 = __shfl_xor(c, o, 64);
    double t, e;
    two_sum(s, s2, t, e);
    s = t;
    c += c2 + e;
  }
  if (lane == 0) {
    sv[wave] = s;
    sc[wave] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double S = 0.0, C = 0.0;
    for (int i = 0; i < nw; ++i) {
      double t, e;
      two_sum(S, sv[i], t, e);
      S = t;
      C += sc[i] + e;
    }
    out[col] = (S + C) * scale;
  }
}

__global__ void __launch_bounds__(256)
    k_finalize_cols(const double* __restrict__ part, int nb, int ncols, double scale,
                    double* __restrict__ out) {
  finalize_col(part, nb, ncols, blockIdx.x, scale, out);
}

// The same for partials stored column after column (put_partial); as many
// lanes as finalize_lanes.
inline int finalize_lanes(int nb) { return nb <= 2048 ? 256 : 1024; }
__global__ void __launch_bounds__(1024)
    k_finalize_rows(const double* __restrict__ part, int nb, double scale,
                    double* __restrict__ out) {
  finalize_col(part + static_cast<size_t>(blockIdx.x) * nb, nb, 1, 0, scale, out + blockIdx.x);
}

}  // namespace
}  // namespace lmm
}  // namespace koo
