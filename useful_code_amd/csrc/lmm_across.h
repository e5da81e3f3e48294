// lmm_across.h -- the predictor-corrector step and its reverse with the rates
// of a path across the lanes of a wavefront, for path counts too small to fill
// the GPU with a path per lane.
//
// A path takes W = 16, 32 or 64 lanes, lane r rate r; its state stays in the
// lane's register.  Within a step a rate needs the others only through the
// sums over the rates below it (above it, in the reverse), which are prefix
// sums over the lanes (DPP additions), so a step costs one rate's chain and the
// scans instead of a chain per alive rate.  It issues about five times the
// vector instructions of a path per lane (scans, dead rates), from W times the
// wavefronts.
#pragma once

#include "lmm_step.h"

namespace koo {
namespace lmm {
namespace {

constexpr int kAcrossLanes = 256;

// Paths of a block.
template <int W>
constexpr int kAcrossBlock = kAcrossLanes / W;

template <int Ctrl, int Rows>
__device__ __forceinline__ float lane_shift(float old, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), Ctrl,
                                                    Rows, 0xf, false));
}
// Sums over this lane and those below it in the path's W lanes, of the F values
// v[0..F): shifts by 1, 2, 4, 8 inside rows of 16, then the row below's last
// lane, then lane 31.  Written as instructions: the compiler takes three for an
// addition under a row mask.  A lane's shifted read needs two wait states after
// the write of the register, which the other registers' additions are.
#define KOO_DPP(op, i) "v_add_f32_dpp %" #i ", %" #i ", %" #i " " op "\n"
#define KOO_SHR(n) "row_shr:" #n " row_mask:0xf bank_mask:0xf bound_ctrl:0"
#define KOO_B15 "row_bcast:15 row_mask:0xa bank_mask:0xf"
#define KOO_B31 "row_bcast:31 row_mask:0xc bank_mask:0xf"
#define KOO_STEP1(op) "s_nop 1\n" KOO_DPP(op, 0)
#define KOO_STEP2(op) "s_nop 0\n" KOO_DPP(op, 0) KOO_DPP(op, 1)
#define KOO_STEP3(op) KOO_DPP(op, 0) KOO_DPP(op, 1) KOO_DPP(op, 2)
#define KOO_STEP4(op) KOO_STEP3(op) KOO_DPP(op, 3)
#define KOO_STEP5(op) KOO_STEP4(op) KOO_DPP(op, 4)
#define KOO_ROW(S) "s_nop 1\n" S(KOO_SHR(1)) S(KOO_SHR(2)) S(KOO_SHR(4)) S(KOO_SHR(8))
#define KOO_SCAN(S, ...)                                                             \
  if constexpr (W == 16) asm(KOO_ROW(S) : __VA_ARGS__);                              \
  else if constexpr (W == 32) asm(KOO_ROW(S) S(KOO_B15) : __VA_ARGS__);              \
  else asm(KOO_ROW(S) S(KOO_B15) S(KOO_B31) : __VA_ARGS__)
template <int W, int F, int N = F>
__device__ __forceinline__ void scan_add(float (&v)[F]) {
  constexpr int o = F - N;  // from here on
  if constexpr (N == 1) {
    KOO_SCAN(KOO_STEP1, "+v"(v[o]));
  } else if constexpr (N == 2) {
    KOO_SCAN(KOO_STEP2, "+v"(v[o]), "+v"(v[o + 1]));
  } else if constexpr (N == 5) {
    KOO_SCAN(KOO_STEP5, "+v"(v[o]), "+v"(v[o + 1]), "+v"(v[o + 2]), "+v"(v[o + 3]), "+v"(v[o + 4]));
  } else if constexpr (N == 4 || N > 6) {
    KOO_SCAN(KOO_STEP4, "+v"(v[o]), "+v"(v[o + 1]), "+v"(v[o + 2]), "+v"(v[o + 3]));
    if constexpr (N > 4) scan_add<W, F, N - 4>(v);
  } else {
    KOO_SCAN(KOO_STEP3, "+v"(v[o]), "+v"(v[o + 1]), "+v"(v[o + 2]));
    if constexpr (N > 3) scan_add<W, F, N - 3>(v);
  }
}
template <int W>
__device__ __forceinline__ float scan_add(float x) {
  float v[1] = {x};
  scan_add<W>(v);
  return v[0];
}
#undef KOO_SCAN
#undef KOO_ROW
#undef KOO_STEP5
#undef KOO_STEP4
#undef KOO_STEP3
#undef KOO_STEP2
#undef KOO_STEP1
#undef KOO_B31
#undef KOO_B15
#undef KOO_SHR
#undef KOO_DPP
template <int W>
__device__ __forceinline__ float scan_mul(float v) {
  v *= lane_shift<0x111, 0xf>(1.0f, v);
  v *= lane_shift<0x112, 0xf>(1.0f, v);
  v *= lane_shift<0x114, 0xf>(1.0f, v);
  v *= lane_shift<0x118, 0xf>(1.0f, v);
  if constexpr (W >= 32) v *= lane_shift<0x142, 0xa>(1.0f, v);
  if constexpr (W == 64) v *= lane_shift<0x143, 0xc>(1.0f, v);
  return v;
}

// This lane's place: rate r of path p (live if there is such a path and rate).
template <int W>
struct AcrossLane {
  int r, p;
  bool rate, live;
  __device__ __forceinline__ AcrossLane(const Model& m, int block)
      : r(threadIdx.x & (W - 1)),
        p(block * kAcrossBlock<W> + static_cast<int>(threadIdx.x) / W),
        rate(r < m.N),
        live(rate && p < m.P) {}
};

// The pseudo-roots of rate r at step s, zero for a rate that is not alive
// (its state and adjoint then pass through the step unchanged): read from the
// step's row as a buffer, dead rates at an offset past its end.
template <int F>
__device__ __forceinline__ void load_roots(const Model& m, int s, int r, bool rate,
                                           float (&a)[F]) {
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(
      (float*)(m.A + static_cast<size_t>(s) * m.N * F), 0, 4 * F * m.N, 0x00027000);
  const int at = rate && r >= s ? 4 * F * r : 0x40000000;
#pragma unroll
  for (int f = 0; f < F; ++f)
    a[f] = __int_as_float(
        static_cast<int>(__builtin_amdgcn_raw_buffer_load_b32(rs, at + 4 * f, 0, 0)));
}

template <int F>
__device__ __forceinline__ float fixed_drift(const float (&a)[F]) {
  float c = 0.0f;
#pragma unroll
  for (int f = 0; f < F; ++f) c = fmaf(a[f], a[f], c);
  return -0.5f * kLog2e * c;
}
template <int F>
__device__ __forceinline__ float dot(const float (&a)[F], const float (&b)[F]) {
  float s = 0.0f;
#pragma unroll
  for (int f = 0; f < F; ++f) s = fmaf(a[f], b[f], s);
  return s;
}

// All N steps of the lanes' paths (pc_step, lmm_step.h, with the sums as
// scans); returns the rate's state as it fixed.  keep(s, x, my, md): the state
// before step s and the step's sums sum_f a y, sum_f a d.
template <int F, int W, class Keep>
__device__ __forceinline__ float across_steps(const Model& m, const AcrossLane<W>& at, float kr,
                                              Keep keep) {
  const int N = m.N;
  // lane s of the path holds the variates of step s
  float zl[F], a[F], an[F], z[F], zn[F];
#pragma unroll
  for (int f = 0; f < F; ++f)
    zl[f] = at.live ? kLog2e * m.z[(static_cast<size_t>(at.r) * F + f) * m.P + at.p] : 0.0f;
  load_roots<F>(m, 0, at.r, at.rate, an);
#pragma unroll
  for (int f = 0; f < F; ++f) zn[f] = __shfl(zl[f], 0, W);
  float x = 0.0f;
  for (int s = 0; s < N; ++s) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
      a[f] = an[f];
      z[f] = zn[f];
    }
    const int next = min(s + 1, N - 1);
    load_roots<F>(m, next, at.r, at.rate, an);
#pragma unroll
    for (int f = 0; f < F; ++f) zn[f] = __shfl(zl[f], next, W);
    const float c = fixed_drift<F>(a);
    const float G = drift_coeff(x, kr);
    float y[F], d[F];
#pragma unroll
    for (int f = 0; f < F; ++f) y[f] = G * a[f];
    scan_add<W>(y);
#pragma unroll
    for (int f = 0; f < F; ++f) y[f] += z[f];
    const float my = dot<F>(a, y);
    const float xh = x + c + my;
    const float g = drift_coeff(xh, kr) - G;
#pragma unroll
    for (int f = 0; f < F; ++f) d[f] = g * a[f];
    scan_add<W>(d);
    const float md = dot<F>(a, d);
    keep(s, x, my, md);
    x = fmaf(0.5f, md, xh);
  }
  return x;
}

// What across_steps keeps for the reverse: per path three triangular arrays in
// LDS (state, sum a y, sum a d), the N - s alive rates of step s from the top
// rate down.  A rate dead at the step reads entries of later steps (at the
// array's end the last one): finite ones, which its zero pseudo-roots cancel.
__host__ __device__ constexpr int across_tri(int N) { return N * (N + 1) / 2; }
__host__ __device__ constexpr int across_tri_row(int N, int s) { return s * N - s * (s - 1) / 2; }

// Reverse of the N steps with the rates from the top down over the lanes (lane
// l rate r = N - 1 - l), so that the sums over the rates above are prefix sums
// too (reverse_step, lmm_step.h).  lam: on entry the adjoint of the state as it
// fixed, on exit that of the initial state; returns the sum of the vega terms.
template <int F, int W, class Kept>
__device__ __forceinline__ float across_reverse(const Model& m, int r, bool rate, float kr,
                                                float& lam, Kept kept) {
  float a[F], an[F], w = 0.0f;
  load_roots<F>(m, m.N - 1, r, rate, an);
  for (int s = m.N - 1; s >= 0; --s) {
#pragma unroll
    for (int f = 0; f < F; ++f) a[f] = an[f];
    load_roots<F>(m, max(s - 1, 0), r, rate, an);
    float x, my, md;
    kept(s, x, my, md);
    const float c = fixed_drift<F>(a);
    const float G = drift_coeff(x, kr);
    const float Gh = drift_coeff(x + c + my, kr);
    const float lh = 0.5f * lam;
    float D[F], Y[F];
#pragma unroll
    for (int f = 0; f < F; ++f) D[f] = lh * a[f];
    scan_add<W>(D);
    const float q = dot<F>(a, D);
    const float uh = Gh * q;
    const float xhb = fmaf(uh, drift_slope(Gh), lam);
#pragma unroll
    for (int f = 0; f < F; ++f) Y[f] = xhb * a[f];
    scan_add<W>(Y);
    const float p = dot<F>(a, Y);
    const float ug = G * (p - q);
    const float term = fmaf(xhb, fmaf(2.0f, c, my), fmaf(lh, md, uh + ug));
    w += r >= s ? term : 0.0f;
    lam = fmaf(ug, drift_slope(G), xhb);
  }
  return w;
}

}  // namespace
}  // namespace lmm
}  // namespace koo
