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
  int P, N, k;
};

// The step table: for every step s and alive rate r >= s the pair
// {fixed drift c = -0.5 log2(e) sum_f A(s,r,f)^2, kr of drift_coeff}, steps one
// after the other (N - s pairs each): N (N + 1) floats.
__host__ __device__ constexpr size_t step_table_floats(int N) {
  return static_cast<size_t>(N) * N + N;
}
// First float of step s.
__host__ __device__ constexpr int step_table_row(int N, int s) { return s * (2 * N + 1 - s); }

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
  t[1] = kLn2 * (1.0f / m.taus[r] - m.disp[r]) / (m.f0[r] + m.disp[r]);
}

// Every lane of the block takes part; the caller then synchronises.
template <int F>
__device__ __forceinline__ void fill_step_table(const Model& m, float* tab) {
  for (int q = threadIdx.x; q < m.N * m.N; q += blockDim.x) put_step_entry<F>(m, q, tab);
}

// A rate's f + d at the start, by which 2^x is scaled.
__device__ __forceinline__ float start_level(const Model& m, int r) { return m.f0[r] + m.disp[r]; }

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
  // `base`: element 0 of the row; on: no lane reads or stores anything if false
  __device__ __forceinline__ PathRow row(const float* base, bool on = true) const {
    return PathRow{__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base) + p0, 0,
                                                     on ? 4 * n : 0, 0x00027000),
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
  __device__ __forceinline__ PathRow row(const float* base, int r, bool on = true) const {
    return row(base + static_cast<size_t>(r) * P, on);
  }
};

// Vega terms of a wavefront, summed over its lanes on the matrix cores: the
// term of the rate j places from the top is the A operand of a 16x16x4 product
// whose B is one in column j mod 16, so column j of tile j / 16 collects 16
// partial sums (of four lanes each) over all steps.  Two issue slots a rate
// (the one-hot column and the product), where folding the 64 lanes by DPP and
// adding to LDS takes about eight.
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
  // out[j] (LDS) = the wavefront's sum of the rate j places from the top
  __device__ __forceinline__ void sums(double* out, int rates) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      double v = (static_cast<double>(acc[t][0]) + static_cast<double>(acc[t][1])) +
                 (static_cast<double>(acc[t][2]) + static_cast<double>(acc[t][3]));
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (lane < 16 && 16 * t + lane < rates) out[16 * t + lane] = v;
    }
  }
};

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
// would carry what only vector instructions use in vector registers).
__device__ __forceinline__ float keep_scalar(float x) {
  int i = __float_as_int(x);
  asm volatile("" : "+s"(i));
  return __int_as_float(i);
}
// A table in LDS is read into vector registers and stays there.
template <int F, int U, class Tab>
__device__ __forceinline__ Rows<F, U> scalar_rows(const Rows<F, U>& v) {
  constexpr bool kScalarTab = std::is_same<Tab, c_cfloat>::value;
  Rows<F, U> w;
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int f = 0; f < F; ++f) w.a[u][f] = keep_scalar(v.a[u][f]);
    w.c[u] = v.c[u];
    w.kr[u] = v.kr[u];
    if constexpr (kScalarTab) {
      w.c[u] = keep_scalar(w.c[u]);
      w.kr[u] = keep_scalar(w.kr[u]);
    }
  }
  return w;
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

// The first window of a step, fetched while the step before it ends.
template <int F, int U>
struct Ahead {
  Rows<F, U> rows;
  float x[U];  // states
  float l[U];  // their adjoints (the reverse)
};

// Fetches the first window of PC step s; `load(r)` gives the state of rate r.
template <int F, int U, class Tab, class Load>
__device__ __forceinline__ void pc_fetch(Ahead<F, U>& h, const Model& m, int s, Tab tab,
                                         Load load) {
  const int base = part_base<U>(m.N, s);
  load_rows<F, U>(h.rows, m, tab, s, base);
#pragma unroll
  for (int i = 0; i < U; ++i) h.x[i] = load(max(base + i, s));
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
  Rows<F, U> w;
  float x[U], first = 0.0f;
  // takes the fetched window and fetches the one at r
  auto take = [&](int r) {
    window_ready();
    w = scalar_rows<F, U, Tab>(h.rows);
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = h.x[u];
    if (r < N) {
      load_rows<F, U>(h.rows, m, tab, s, r);
#pragma unroll
      for (int u = 0; u < U; ++u) h.x[u] = load(r + u);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int base = part_base<U>(N, s), end = part_end<U>(N, s);
  take(end);
#pragma unroll
  for (int i = 0; i < U; ++i)
    if (base + i >= s && base + i < end) {
      const float v = rate(w, i, x[i], base + i);
      if (base + i == s) first = v;
    }
  for (int r0 = end; r0 < N; r0 += U) {
    take(r0 + U);
#pragma unroll
    for (int u = 0; u < U; ++u) rate(w, u, x[u], r0 + u);
  }
  return first;
}

// Fetches the first window of the reverse of step s (rates N-1, N-2, ...): a
// full one, or the one with rate s.
template <int F, int U, class Tab, class Src, class Lam>
__device__ __forceinline__ void reverse_fetch(Ahead<F, U>& h, const Model& m, int s, Tab tab,
                                              Src src, const Lam& lam) {
  load_rows<F, U>(h.rows, m, tab, s, m.N - U);
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const int r = max(m.N - U + i, s);
    h.x[i] = src(r);
    h.l[i] = lam.get(r);
  }
}

// Reverse of PC step s over the rates N-1..s.  On entry `lam.get(r)` holds the
// adjoint of the end-of-step state r, on exit that of the start-of-step one
// (`lam.set`).  `h`: reverse_fetch of this step.  y / d are the step's final
// sums (un-accumulated here); `src(r)` gives the start state of rate r.
// `fixing(lp, x')` adds the product's adjoint of the rate fixing at the end of
// the step (r == s) to lp; `vegas` takes w = sum_f Abar(s,r,f) A(s,r,f) of the
// step, which contracts to scalars the reverse already has: with the adjoint
// sums D of d and Y of y (rates descending),
//   D_f += 0.5 lp a_f, q = sum a D;   xhb = lp + q dGh/dx
//   Y_f += xhb a_f,    p = sum a Y;   lam = xhb + (p - q) dG/dx
//   w = 0.5 lp sum a d + (Gh - G) q + G p + xhb (sum a y + 2 c).
template <int F, int U, class Tab, class Src, class Lam, class Fixing, class Vegas>
__device__ __forceinline__ void reverse_step(const Model& m, int s, Tab tab, Ahead<F, U>& h,
                                             Src src, const Lam& lam, float (&y)[F],
                                             float (&d)[F], Fixing fixing, Vegas& vegas) {
  const int N = m.N;
  float D[F], Y[F];
#pragma unroll
  for (int f = 0; f < F; ++f) D[f] = Y[f] = 0.0f;
  auto rate = [&](const Rows<F, U>& v, int u, float x, float lp, int r, bool may_fix) {
    const float c = v.c[u];
    const float G = drift_coeff(x, v.kr[u]);
    float my = 0.0f, md = 0.0f;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      my = fmaf(v.a[u][f], y[f], my);
      md = fmaf(v.a[u][f], d[f], md);
    }
    const float mc = my + c;
    const float xh = x + mc;
    const float Gh = drift_coeff(xh, v.kr[u]);
    if (may_fix && r == s) fixing(lp, fmaf(0.5f, md, xh));
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
    return fmaf(xhb, mc + c, fmaf(lh, md, uh + ug));
  };
  Rows<F, U> v;
  float x[U], l[U];
  // takes the fetched window; then fetches the one at r, if any
  auto take = [&](bool more, int r) {
    window_ready();
    v = scalar_rows<F, U, Tab>(h.rows);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      x[i] = h.x[i];
      l[i] = h.l[i];
    }
    if (more) {
      load_rows<F, U>(h.rows, m, tab, s, r);
#pragma unroll
      for (int i = 0; i < U; ++i) {
        h.x[i] = src(max(r + i, s));
        h.l[i] = lam.get(max(r + i, s));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int base = part_base<U>(N, s), end = part_end<U>(N, s);
  // full windows [r0, r0 + U); the window after the last of them is at base
  for (int r0 = N - U; r0 >= end; r0 -= U) {
    take(true, r0 - U >= end ? r0 - U : base);
    float w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = rate(v, U - 1 - u, x[U - 1 - u], l[U - 1 - u], r0 + U - 1 - u, false);
    vegas.add(N - U - r0, w);
  }
  // the window with rate s
  take(false, 0);
#pragma unroll
  for (int i = U - 1; i >= 0; --i)
    if (base + i >= s && base + i < end) {
      const float w[1] = {rate(v, i, x[i], l[i], base + i, true)};
      vegas.add(N - 1 - base - i, w);
    }
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
      xn[i] = X.get(max(r + i, s));
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

// Tiles of VegaSums: blocks of 256 lanes take up to 45 rates, those of one
// wavefront up to kMaxRates.
template <int BD>
constexpr int kVegaTiles = BD == 256 ? 3 : (kMaxRates + 15) / 16;

// A block's sums of the state adjoints (rows of BD lanes in LDS) and vega
// terms, as deltas (d/df0_r = log2(e) lam_r / (f0_r + d_r)) and vegas (over
// sigma_r) into out[0..N) and out[N..2N).  Overwrites the LDS rows.  Agent: the
// stores are agent-coherent.
template <int BD, bool Agent = false, class Vegas>
__device__ __forceinline__ void adjoint_sums(const Model& m, const float* __restrict__ vols,
                                             float* lds, const Vegas& vegas, double* out) {
  const int N = m.N, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int W = BD / 64;
  auto put = [&](double* o, double v) {
    if (Agent) store_agent(o, v);
    else *o = v;
  };
  __syncthreads();
  // a wavefront sums whole rows
  for (int r = wave; r < N; r += W) {
    double v = 0.0;
#pragma unroll
    for (int i = 0; i < W; ++i) v += static_cast<double>(lds[r * BD + 64 * i + lane]);
    v = wave_sum_f64(v);
    if (lane == 0)
      put(out + r, v * static_cast<double>(kLog2e) / static_cast<double>(start_level(m, r)));
  }
  __syncthreads();
  double* red = reinterpret_cast<double*>(lds);  // [W][N]
  vegas.sums(red + wave * N, N);
  __syncthreads();
  for (int j = threadIdx.x; j < N; j += BD) {
    double v = 0.0;
#pragma unroll
    for (int i = 0; i < W; ++i) v += red[i * N + j];
    const int r = N - 1 - j;
    put(out + N + r, v / static_cast<double>(vols[r]));
  }
}

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

// The model arrays are separate __restrict__ kernel arguments (not members of
// a by-value struct) so the compiler may read them through the scalar cache.
#define KOO_MODEL_PARAMS                                                                  \
  const float* __restrict__ z_, const float* __restrict__ f0_,                            \
      const float* __restrict__ taus_, const float* __restrict__ disp_,                   \
      const float* __restrict__ A_, float strike_, int P_, int N_, int k_
#define KOO_MODEL_LOCAL \
  const Model m{z_, cmem(f0_), cmem(taus_), cmem(disp_), cmem(A_), strike_, P_, N_, k_}

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

// Rate-count class of a product in a batched portfolio (launches are per
// class so LDS is reserved for the class's largest curve).
inline int rate_class(int rates) { return rates <= 16 ? 0 : (rates <= 24 ? 1 : (rates <= 32 ? 2 : 3)); }

// out[col] = (sum_b part[b*ncols + col]) * scale, compensated; called by a
// whole block (k_finalize_cols runs one block per column).  Agent: the
// partials are read with agent-coherent loads.
template <bool Agent = false>
__device__ __forceinline__ void finalize_col(const double* __restrict__ part, int nb, int ncols,
                                             int col, double scale, double* __restrict__ out) {
  __shared__ double sv[16], sc[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  // per lane: Neumaier over a strided slice of the blocks
  double s = 0.0, c = 0.0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    const double x = Agent ? load_agent(part + static_cast<size_t>(b) * ncols + col)
                           : part[static_cast<size_t>(b) * ncols + col];
    const double t = s + x;
    c += (fabs(s) >= fabs(x)) ? (s - t) + x : (x - t) + s;
    s = t;
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

}  // namespace
}  // namespace lmm
}  // namespace koo
