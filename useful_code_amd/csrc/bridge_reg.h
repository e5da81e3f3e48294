// bridge_reg.h -- the Brownian bridge with a lane's points in registers, shared
// by the stand-alone bridge and the fused generator.
#pragma once

#include <utility>

#include "bridge_device.h"

namespace koo {
namespace {

// ---------------------------------------------------------------------------
// Register-resident bridge (stand-alone for S <= kRegSteps, the generator for
// every S).  The construction order depends on S only, so for a compile-time S
// every index is a constant and the S bridge points of a lane stay in VGPRs (no
// LDS path storage, which held occupancy to one or two waves per SIMD).  The
// stand-alone bridge reads its weights from the kernel arguments (uniform,
// scalar loads); the fused generator, which loops over chunks, from an LDS copy
// (LdsWeights).
// ---------------------------------------------------------------------------
constexpr int kRegSteps = 64;

// The index walk of make_tables (brownian_bridge.cu:639-700) as a constant
// expression.
template <int S>
struct BridgeOrder {
  int16_t bridge[S] = {}, left[S] = {}, right[S] = {};
  constexpr BridgeOrder() {
    int map[S] = {};
    map[S - 1] = 1;
    bridge[0] = S - 1;
    for (int j = 0, i = 1; i < S; ++i) {
      while (map[j]) ++j;
      int k = j;
      while (!map[k]) ++k;
      const int l = j + ((k - 1 - j) >> 1);
      map[l] = i;
      bridge[i] = static_cast<int16_t>(l);
      left[i] = static_cast<int16_t>(j);
      right[i] = static_cast<int16_t>(k);
      j = k + 1;
      if (j >= S) j = 0;
    }
  }
};

// V is float (one path), f32x2 or f32x4 (two, four paths; the scalar weights
// broadcast).
template <int S, int I, class V, class Z, class W>
__device__ __forceinline__ void bridge_point(V (&w)[S], const W& wt, Z& z) {
  constexpr BridgeOrder<S> M{};
  float rw, lw, sd;
  wt.get(I, rw, lw, sd);
  if constexpr (I == 0) {
    w[S - 1] = sd * z(0);
  } else {
    constexpr int j = M.left[I], k = M.right[I], l = M.bridge[I];
    V v = rw * w[k];
    if constexpr (j != 0) v = bridge_fma(lw, w[j - 1], v);
    w[l] = bridge_fma(sd, z(I), v);
  }
}

template <int S, class V, class Z, class W, int... I>
__device__ __forceinline__ void bridge_points(V (&w)[S], const W& wt, Z& z,
                                              std::integer_sequence<int, I...>) {
  (bridge_point<S, I>(w, wt, z), ...);
}

// In-place form for variates that come from memory: w[bridge(i)] holds
// variate i on entry (so all S loads can be in flight at once, into the
// registers the points end in), and point bridge(i) replaces it; the same
// operations in the same order as bridge_point.
template <int S, int I, class V>
__device__ __forceinline__ void bridge_point_inplace(V (&w)[S], const BridgeTables& T) {
  constexpr BridgeOrder<S> M{};
  if constexpr (I == 0) {
    w[S - 1] = T.sd[0] * w[S - 1];
  } else {
    constexpr int j = M.left[I], k = M.right[I], l = M.bridge[I];
    V v = T.rw[I] * w[k];
    if constexpr (j != 0) v = bridge_fma(T.lw[I], w[j - 1], v);
    w[l] = bridge_fma(T.sd[I], w[l], v);
  }
}

template <int S, class V, class Load, int... I>
__device__ __forceinline__ void bridge_points_loaded(V (&w)[S], const BridgeTables& T,
                                                     Load load,
                                                     std::integer_sequence<int, I...>) {
  constexpr BridgeOrder<S> M{};
  ((w[M.bridge[I]] = load(I)), ...);
  (bridge_point_inplace<S, I>(w, T), ...);
}

}  // namespace
}  // namespace koo
