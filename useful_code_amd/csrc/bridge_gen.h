// bridge_gen.h -- the fused Sobol -> scramble -> normal -> bridge generator
// kernel.  Its instances, one for each step count, are compiled in four files
// (bridge_gen_*.hip) side by side: in one they took four minutes.
#pragma once

#include <array>
#include <type_traits>

#include "bridge_reg.h"

namespace koo {

// The kernel for `steps` steps, kBridgeGenFirst[part] <= steps <
// kBridgeGenFirst[part + 1], to launch with the arguments of
// k_sobol_bridge_reg; parts are cut so that they compile in about the same time.
constexpr int kBridgeGenParts = 4;
constexpr int kBridgeGenFirst[kBridgeGenParts + 1] = {1, 65, 91, 111, 129};
const void* bridge_gen_kernel_0(int steps);
const void* bridge_gen_kernel_1(int steps);
const void* bridge_gen_kernel_2(int steps);
const void* bridge_gen_kernel_3(int steps);

namespace {

static_assert(kBridgeGenFirst[kBridgeGenParts] == kBridgeMaxSteps + 1, "every step count");

// The construction weights of step i, {rw, lw, sd}, from a copy of the
// tables in LDS ({rw, lw, sd, 0} per step) read at an index offset the
// compiler cannot see through.  A loop over chunks that reads the
// kernel-argument tables gets all 3 S weights hoisted into scalar registers,
// more than there are (spilled through vector lanes); the LDS copy is read
// where each weight is used.
struct LdsWeights {
  const f32x4* w;  // LDS
  int z;           // zero, opaque to the compiler
  __device__ __forceinline__ void get(int i, float& rw, float& lw, float& sd) const {
    const f32x4 q = w[i + z];
    rw = q.x;
    lw = q.y;
    sd = q.z;
  }
};

// Fused generator on the register bridge, every step count.  Each wavefront
// walks a contiguous run of 64-path chunks of one factor, two at a time and an
// odd last one alone.  With n = G + l (G a multiple of 64, l < 64) the Gray code
// splits, gray(n) = gray(G) ^ gray(l), so the scrambled Sobol integer is
// X(G) ^ T(l) with X(G) = scrambler ^ XOR of the direction numbers over the set
// bits of gray(G).  A lane's l is the same in every chunk; T(l) sits in LDS.
// X(G) is kept one dimension per lane (two registers beyond 64 steps): from
// G = 64m to 64(m+1) gray flips bits 5 and 6 + ctz(m+1), so advancing costs two
// XORs.  A chunk (lanes at n = 64c + off1 + lane) spans G and G + 64, two chunks
// three values: the wavefront writes them to rows of its own in LDS, from which
// each lane reads those of its group, four dimensions to a read.
// Bound by the vector instructions, 26 a point, most of them the quantile; 43
// with one chunk at a time, X(G) read out by readlane and 64-bit store
// addresses.  2^20 paths: 40 steps x 5 factors 232 -> 175 us, 64 x 32 2.59 ->
// 1.93 ms (4.4 TB/s of stores).  Step counts above 64 kept the points in LDS
// and walked the bits of the Gray code for each: 2^17 x 80 x 2 238 -> 43 us.
// Few paths leave a wavefront one chunk: in a pair half of that is for nothing
// (65536 paths x 32 x 5 24.6 us, 18.4 alone; 4096 x 40 x 8 12.2, 10.4).  Beyond
// kRegSteps the body for one chunk is left out: those kernels take most of the
// library's compile time.
template <int S>
__global__ void __launch_bounds__(kBridgeThreads)
    k_sobol_bridge_reg(const BridgeTables T, int factors, int paths, uint32_t off1,
                       const uint32_t* __restrict__ dirs, const uint32_t* __restrict__ scr,
                       int number_scrambled, const int* __restrict__ alloc,
                       float* __restrict__ out) {
  constexpr int R = (S + 63) / 64;  // dimensions per lane in the X(G) bookkeeping
  constexpr int Q = (S + 3) / 4;    // groups of four dimensions
  __shared__ uint32_t vall[S * 32];                      // direction numbers [bridge variate][bit]
  __shared__ u32x4 tlo[Q * 64];                          // T(l) [group][l]
  __shared__ u32x4 xrows[(kBridgeThreads / 64) * 3 * Q]; // X(G), X(G+64), X(G+128) per wavefront
  __shared__ f32x4 wts[S];                               // construction weights {rw, lw, sd, 0}
  const int f = blockIdx.y;
  const int* idx = alloc + f * S;
  for (int q = threadIdx.x; q < S * 32; q += blockDim.x)
    vall[q] = dirs[static_cast<size_t>(idx[q >> 5]) * 32 + (q & 31)];
  for (int q = threadIdx.x; q < S; q += blockDim.x) wts[q] = f32x4{T.rw[q], T.lw[q], T.sd[q], 0.0f};
  __syncthreads();
  for (int q = threadIdx.x; q < S * 64; q += blockDim.x) {
    const uint32_t l = static_cast<uint32_t>(q & 63), g = l ^ (l >> 1);
    const uint32_t* vv = vall + (q >> 6) * 32;
    uint32_t x = 0;
#pragma unroll
    for (int bit = 0; bit < 6; ++bit)
      if ((g >> bit) & 1u) x ^= vv[bit];
    reinterpret_cast<uint32_t*>(tlo)[(q >> 8) * 256 + l * 4 + ((q >> 6) & 3)] = x;
  }
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x >> 6);
  const int64_t wv = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + wave;
  const int64_t chunks = (static_cast<int64_t>(paths) + 63) >> 6;
  // scalars: the loop below and its addresses are uniform
  const int c0 = __builtin_amdgcn_readfirstlane(static_cast<int>(wv * chunks / waves));
  const int c1 = __builtin_amdgcn_readfirstlane(static_cast<int>((wv + 1) * chunks / waves));
  if (c0 >= c1) return;

  const uint32_t r = off1 & 63u;
  const uint32_t l = (r + static_cast<uint32_t>(lane)) & 63u;
  uint32_t m = static_cast<uint32_t>(c0) + (off1 >> 6);  // G = 64 m for chunk c0
  // this lane's dimensions for the X(G) bookkeeping
  const uint32_t* vd[R];
  uint32_t x[R], v5[R];
  uint32_t* xw = reinterpret_cast<uint32_t*>(xrows + wave * 3 * Q) + lane;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int dl = 64 * k + lane < S ? 64 * k + lane : S - 1;
    vd[k] = vall + dl * 32;
    const int d = idx[dl];
    x[k] = d < number_scrambled ? scr[d] : 0u;
    const uint32_t G = m << 6, g = G ^ (G >> 1);
    for (int b = 5; b < 32; ++b)
      if ((g >> b) & 1u) x[k] ^= vd[k][b];
    v5[k] = vd[k][5];
  }
  auto put = [&](int row) {
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (64 * k + lane < S) xw[row * 4 * Q + 64 * k] = x[k];
  };
  // bits 5 and t of gray, t = 6 + ctz of the next m
  auto advance = [&] {
    const int t = 6 + __builtin_ctz(++m);
#pragma unroll
    for (int k = 0; k < R; ++k) x[k] ^= v5[k] ^ (t < 32 ? vd[k][t] : 0u);
  };
  const u32x4* tl = tlo + l;
  // the lane's own group of the first chunk; of the second, a row further
  const u32x4* xl = xrows + wave * 3 * Q + (r + static_cast<uint32_t>(lane) >= 64u ? Q : 0);
  // the wavefront's paths as a buffer per step: stores past its last path are
  // dropped (lanes past the last path; the second chunk of a last pair)
  const int bytes = 4 * min(paths - c0 * 64, (c1 - c0) * 64);
  float* first = out + static_cast<size_t>(f) * paths + static_cast<size_t>(c0) * 64;
  // `chunks`: two at a time, or one
  auto walk = [&](int c, auto chunks) {
    constexpr bool two = decltype(chunks)::value == 2;
    using V = typename std::conditional<two, f32x2, float>::type;
    // a wavefront's LDS operations keep their order, and the rows are its own
    put(0);
    advance();
    put(1);
    if constexpr (two) {
      advance();
      put(2);
    }
    __builtin_amdgcn_wave_barrier();
    u32x4 t, a, b;
    auto z = [&](int i) {
      if (i % 4 == 0) {
        t = tl[(i >> 2) * 64];
        a = xl[i >> 2];
        if constexpr (two) b = xl[Q + (i >> 2)];
      }
      const float first = invnorm_u32(t[i & 3] ^ a[i & 3]);
      if constexpr (two) return f32x2{first, invnorm_u32(t[i & 3] ^ b[i & 3])};
      else return first;
    };
    // The weights come from LDS at an offset, and the rows of the steps from a
    // stride, made opaque each time (a zero from s_mov), so that their reads
    // and sums stay in the loop.
    int zero;
    asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
    V w[S];
    const LdsWeights wt{wts, zero};
    bridge_points<S>(w, wt, z, std::make_integer_sequence<int, S>{});
    const size_t stride = (static_cast<size_t>(factors) + zero) * paths;
    float* row = first;
    const int byte = (c - c0) * 256 + lane * 4;
    V prev{};
#pragma unroll
    for (int i = 0; i < S; ++i, row += stride) {
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(row, 0, bytes, 0x00027000);
      const V dz = w[i] - prev;
      if constexpr (two) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dz.x), rs, byte, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dz.y), rs, byte + 256, 0, 0);
      } else {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dz), rs, byte, 0, 0);
      }
      prev = w[i];
    }
    __builtin_amdgcn_wave_barrier();
  };
  int c = c0;
  if constexpr (S <= kRegSteps) {
    for (; c + 1 < c1; c += 2) walk(c, std::integral_constant<int, 2>{});
    if (c < c1) walk(c, std::integral_constant<int, 1>{});
  } else {
    for (; c < c1; c += 2) walk(c, std::integral_constant<int, 2>{});
  }
}

template <int First, int... I>
const void* gen_kernel(int steps, std::integer_sequence<int, I...>) {
  static const std::array<const void*, sizeof...(I)> table{
      reinterpret_cast<const void*>(&k_sobol_bridge_reg<First + I>)...};
  return table[steps - First];
}
// Of a part's own file.
template <int Part>
const void* gen_kernel(int steps) {
  constexpr int first = kBridgeGenFirst[Part], n = kBridgeGenFirst[Part + 1] - first;
  return gen_kernel<first>(steps, std::make_integer_sequence<int, n>{});
}

}  // namespace
}  // namespace koo
