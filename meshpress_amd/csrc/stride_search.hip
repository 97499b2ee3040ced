// Encoder search kernels for gfx950.
//
//  * stream costs / selection: 16 lanes per residual stream (64 for long
//    ones); each lane folds its values into the 20 candidate body costs (Rice k = 0..11, Exp-Golomb
//    k = 0..7, residual_entropy.py:39-54 exact integer form), then a sum over
//    the lanes and the tie-break of _pick_best_k
//    (paradelta_v5_dup.py:159-171, paradelta_codec.py:131-146).
//  * IRLP candidate cost: candidates x slices of a meshlet's samples over the
//    lanes of a wave; each lane evaluates the parallelogram residuals of its
//    candidate on its slice and the 20 coder costs; the slices' sums give the
//    meshlet's cheapest coder, which the wave adds up over its meshlets
//    (_cost_seeds_njit, encoder/_irlp_fit.py:120-183).
//
// Both are bound by VALU issue: 20 coder costs a value.  They run in 32 bits
// wherever a bound taken from the values themselves shows that nothing
// wraps, else in 64.  Measured, 64 bits and a lane per candidate or a wave per
// stream throughout -> now: 60 candidates on 4,000 meshlets 159 -> 66 us, one
// candidate on 17,500 meshlets 170 -> 26 us, 13,500 streams 42 -> 14 us.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "../../include/stride_hip.h"
#include "stride_err.h"

namespace stride {

constexpr int kRiceK = 12;
constexpr int kEgK = 8;
constexpr int kCoders = kRiceK + kEgK;

__device__ __forceinline__ uint32_t zz32(int32_t r) {
  return r < 0 ? ((uint32_t)(-(int64_t)r) << 1) - 1u : ((uint32_t)r << 1);
}
__device__ __forceinline__ uint64_t zz64(int64_t r) {
  return r < 0 ? ((uint64_t)(-r) << 1) - 1u : ((uint64_t)r << 1);
}
// The 20 sums in 64 bits: u >> k for Rice(k); for Exp-Golomb(k) the leading
// zeros of u + 2^k, since floor(log2((u >> k) + 1)) = 63 - k - clz(u + 2^k)
// (coder_sum).  u + 2^7 has to fit 64 bits.
__device__ __forceinline__ void accumulate(uint64_t u, uint64_t (&acc)[kCoders]) {
#pragma unroll
  for (int k = 0; k < kRiceK; ++k) acc[k] += u >> k;
#pragma unroll
  for (int k = 0; k < kEgK; ++k) acc[kRiceK + k] += (uint32_t)__builtin_clzll(u + (1ull << k));
}
// coder j's sum of body bits without its 1 + k a value, from accumulate's sum over n values
__device__ __forceinline__ uint64_t coder_sum(int j, uint64_t acc, uint64_t n) {
  return j < kRiceK ? acc : 2ull * (n * (uint64_t)(63 - (j - kRiceK)) - acc);
}

// Sum over the lanes of a group of `G` lanes that share lane % STEP (powers
// of two).
template <int STEP, int G, class T>
__device__ __forceinline__ T group_sum(T v) {
  if constexpr (STEP == 1 && G == 16 && sizeof(T) == 4) {
    // within a row of 16 by DPP adds: lanes ^ 1, ^ 2, then mirrored halves
    // and rows (their quads are uniform by then)
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true);
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true);
    return v;
  }
#pragma unroll
  for (int o = STEP; o < G; o <<= 1) {
    if constexpr (sizeof(T) == 8) {
      const uint32_t lo = __shfl_xor((uint32_t)v, o, 64);
      const uint32_t hi = __shfl_xor((uint32_t)((uint64_t)v >> 32), o, 64);
      v += (T)(((uint64_t)hi << 32) | lo);
    } else {
      v += __shfl_xor(v, o, 64);
    }
  }
  return v;
}

// Body bits of candidate j for n values given the accumulated sum.
__device__ __forceinline__ uint64_t body_bits(int j, uint64_t acc, uint64_t n) {
  if (j < kRiceK) return acc + n * (uint64_t)(1 + j);
  const int k = j - kRiceK;
  return acc + n * (uint64_t)(1 + k);
}

// The 20 sums in 32 bits, two values at a time (a shift each and one
// three-operand add).  An Exp-Golomb sum counts leading zeros:
// floor(log2((u >> k) + 1)) = 31 - k - clz(u + 2^k), which is 0 for u = 0, so
// a slot without a value adds u = 0.
struct Costs32 {
  uint32_t rice[kRiceK], zeros[kEgK];
  uint32_t slots;   // values added, empty slots among them
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int k = 0; k < kRiceK; ++k) rice[k] = 0;
#pragma unroll
    for (int k = 0; k < kEgK; ++k) zeros[k] = 0;
    slots = 0;
  }
  __device__ __forceinline__ void add2(uint32_t u, uint32_t v) {
#pragma unroll
    for (int k = 0; k < kRiceK; ++k) rice[k] += (u >> k) + (v >> k);
#pragma unroll
    for (int k = 0; k < kEgK; ++k)
      zeros[k] += (uint32_t)__builtin_clz(u + (1u << k)) + (uint32_t)__builtin_clz(v + (1u << k));
    slots += 2;
  }
  // use(j, body cost) of n values; sum(x) adds x up over the lanes that hold them
  template <class Sum, class Use>
  __device__ __forceinline__ void totals(uint64_t n, Sum&& sum, Use&& use) {
    slots = sum(slots);
#pragma unroll
    for (int k = 0; k < kRiceK; ++k) use(k, body_bits(k, sum(rice[k]), n));
#pragma unroll
    for (int k = 0; k < kEgK; ++k) {
      const uint32_t logs = slots * (uint32_t)(31 - k) - sum(zeros[k]);
      use(kRiceK + k, body_bits(kRiceK + k, 2ull * logs, n));
    }
  }
};
// n values of at most umax each: no sum of Costs32 wraps, no addend u + 2^k.
// (Tested by each lane with the largest value it has seen; the wave goes on in
// 32 bits when all of them pass.)
__device__ __forceinline__ bool fits_costs32(uint64_t n, uint64_t umax) {
  return n < (1u << 25) && umax < 0x80000000ull && (umax + 1) * n < 0x80000000ull;
}

// A mesh's streams average 15 to 115 values: four a wave, 16 lanes each.  Where
// one of a wave's four is longer than kLongStream values all 64 lanes share a
// stream: the wave takes the four in turn, or, up to kSpreadStreams streams,
// whose waves do not fill the chip, the workgroup holds four waves for four
// streams and each takes one (three of them end at once otherwise: 0.5 us at
// 8,190 streams, 1.7 at 12,288).  Measured, against 16 lanes whatever the length
// and a wave a stream in 64 bits: one stream of 4,000 values 18 us, 54 and 21;
// 4,000 streams of 1,300 values 30, 89 and 40; 12,288 of them 66 (in turn 103),
// 154 and 101; 13,500 in turn 105, 167 and 107; 54,000 short ones 24, 25, 137.
constexpr int kStreamLanes = 16;
constexpr int64_t kSpreadStreams = 12288, kLongStream = 1024;

// Stream s, the values [b, e), by a group of G lanes; s < 0: no stream, the
// lanes take part in the sums with no values.
template <int G>
__device__ __forceinline__ void stream_cost(const int32_t* __restrict__ vals, int64_t s, int64_t b,
                                            int64_t e, int64_t* __restrict__ costs,
                                            uint8_t* __restrict__ tagk,
                                            int64_t* __restrict__ best_bits) {
  const int lane = threadIdx.x % G;
  const uint64_t n = (uint64_t)(e - b);
  uint32_t bits = 0;
  for (int64_t i = b + lane; i < e; i += G) bits |= zz32(vals[i]);
  const uint64_t umax = bits ? (2ull << (31 - __builtin_clz(bits))) - 1 : 0;
  auto sum = [](auto v) { return group_sum<1, G>(v); };
  uint64_t tot[kCoders];
  if (__all(fits_costs32(n, umax))) {
    Costs32 acc;
    acc.clear();
    for (int64_t i = b + lane; i < e; i += 2 * G) {
      const uint32_t u = zz32(vals[i]);
      const uint32_t v = i + G < e ? zz32(vals[i + G]) : 0u;
      acc.add2(u, v);
    }
    acc.totals(n, sum, [&](int j, uint64_t t) { tot[j] = t; });
  } else {
    uint64_t acc[kCoders];
#pragma unroll
    for (int j = 0; j < kCoders; ++j) acc[j] = 0;
    for (int64_t i = b + lane; i < e; i += G) accumulate(zz32(vals[i]), acc);
#pragma unroll
    for (int j = 0; j < kCoders; ++j) tot[j] = body_bits(j, coder_sum(j, sum(acc[j]), n), n);
  }
  if (lane == 0 && s >= 0) {
    if (costs) {
#pragma unroll
      for (int j = 0; j < kCoders; ++j) costs[s * kCoders + j] = (int64_t)tot[j];
    }
    if (tagk) {
      int rk = 0, ek = 0;
      uint64_t rb = tot[0], eb = tot[kRiceK];
#pragma unroll
      for (int k = 1; k < kRiceK; ++k)
        if (tot[k] < rb) { rb = tot[k]; rk = k; }
#pragma unroll
      for (int k = 1; k < kEgK; ++k)
        if (tot[kRiceK + k] < eb) { eb = tot[kRiceK + k]; ek = k; }
      if (n == 0) { rb = 0; eb = 0; rk = 0; ek = 0; }
      const bool rice = rb <= eb;
      tagk[2 * s] = rice ? 1 : 2;
      tagk[2 * s + 1] = (uint8_t)(rice ? rk : ek);
      if (best_bits) best_bits[s] = (int64_t)(rice ? rb : eb);
    }
  }
}

template <bool SPREAD>
__global__ __launch_bounds__(256) void stream_cost_kernel(const int32_t* __restrict__ vals,
                                                             const int64_t* __restrict__ off,
                                                             int64_t n_streams,
                                                             int64_t* __restrict__ costs,
                                                             uint8_t* __restrict__ tagk,
                                                             int64_t* __restrict__ best_bits) {
  constexpr int G = kStreamLanes, W = 64 / G;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // the wave's first stream, and the lane's
  const int64_t s0 = SPREAD ? W * (int64_t)blockIdx.x : W * (4 * (int64_t)blockIdx.x + wave);
  const int64_t s = s0 + (threadIdx.x & 63) / G;
  const bool some = s < n_streams;
  const int64_t b = some ? off[s] : 0, e = some ? off[s + 1] : 0;
  if (__builtin_expect(!__any(e - b > kLongStream), 1)) {
    if (!SPREAD || wave == 0) stream_cost<G>(vals, some ? s : -1, b, e, costs, tagk, best_bits);
    return;
  }
  const int64_t q1 = s0 + W < n_streams ? s0 + W : n_streams;
#pragma unroll 1
  for (int64_t q = SPREAD ? s0 + wave : s0; q < q1; q += SPREAD ? W : 1)
    stream_cost<64>(vals, q, off[q], off[q + 1], costs, tagk, best_bits);
}

static hipError_t launch_streams(const int32_t* vals, const int64_t* off, int64_t n_streams,
                                 int64_t* costs, uint8_t* tagk, int64_t* best_bits, hipStream_t st) {
  const bool spread = n_streams <= kSpreadStreams;
  const int64_t per = spread ? 4 : 16;
  hipLaunchKernelGGL(spread ? stream_cost_kernel<true> : stream_cost_kernel<false>,
                     dim3((unsigned)((n_streams + per - 1) / per)), dim3(256), 0, st, vals, off,
                     n_streams, costs, tagk, best_bits);
  return hipGetLastError();
}

// A wave's lanes are CB candidates x SL slices x MB meshlets (lane = (meshlet
// SL + slice) CB + candidate), CB the smallest power of two that holds the
// candidates (64 at most, then blocks of 64 along y), SL 16 at most: a lane
// per candidate alone leaves 54 of 64 lanes idle on a fit's 10 seeds and 63
// on its last check.  A wave walks meshlets `gridDim.x` waves apart and adds
// their costs in a register, so that a candidate's total takes one atomic a
// workgroup.
constexpr int kIrlpWaves = 4;

template <int CB, int SL, int MB>
__global__ __launch_bounds__(64 * kIrlpWaves) void irlp_cost_kernel(
    const int32_t* __restrict__ A, const int32_t* __restrict__ B, const int32_t* __restrict__ C,
    const int32_t* __restrict__ Vv, const int64_t* __restrict__ off, int64_t n_m,
    const int32_t* __restrict__ cand, int S, int K, unsigned long long* __restrict__ cost,
    int64_t* __restrict__ per_m) {
  static_assert(CB * SL * MB == 64, "the lanes of a wave");
  constexpr int G = CB * SL;   // lanes a meshlet
  __shared__ unsigned long long part[kIrlpWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int c = lane % CB, slice = (lane / CB) % SL;
  const int sc = blockIdx.y * CB + c;
  const int sr = sc < S ? sc : 0;   // lanes past the last candidate repeat the first
  const int32_t n0 = cand[3 * sr], n1 = cand[3 * sr + 1], n2 = cand[3 * sr + 2];
  const int64_t half = K ? ((int64_t)1 << (K - 1)) : 0;
  auto mag = [](int32_t x) { return (uint64_t)(x < 0 ? -(int64_t)x : (int64_t)x); };
  uint64_t weight = mag(n0) + mag(n1) + mag(n2);   // the largest of the wave's candidates
#pragma unroll
  for (int o = 1; o < CB; o <<= 1) {
    const uint64_t w = ((uint64_t)__shfl_xor((uint32_t)(weight >> 32), o, 64) << 32) |
                       __shfl_xor((uint32_t)weight, o, 64);
    weight = w > weight ? w : weight;
  }
  unsigned long long sum = 0;
#pragma unroll 1
  for (int64_t g = ((int64_t)blockIdx.x * kIrlpWaves + wave) * MB; g < n_m;
       g += (int64_t)gridDim.x * kIrlpWaves * MB) {
    const int64_t m = g + lane / G;
    const int64_t b = m < n_m ? off[m] : 0, e = m < n_m ? off[m + 1] : 0;
    const uint64_t n = (uint64_t)(e - b);
    const int32_t *a0 = A + b, *b0 = B + b, *c0 = C + b, *v0 = Vv + b;
    // bits of the magnitudes among the codes the lane looks at
    uint32_t bits = 0;
    for (uint64_t i = lane % G; i < n; i += G) {
      const int32_t x = a0[i], y = b0[i], z = c0[i], v = v0[i];
      bits |= (uint32_t)((x ^ (x >> 31)) | (y ^ (y >> 31)) | (z ^ (z >> 31)) | (v ^ (v >> 31)));
    }
    const uint64_t top = bits ? (2ull << (31 - __builtin_clz(bits))) : 1;   // |code| <= top
    // 24-bit factors, the weighted sum in 31 bits, and a residual's zigzag
    // value below 2 (top + |prediction| + 1)
    const uint64_t peak = weight * top + (uint64_t)half;
    const bool small = top < (1u << 23) && weight < (1u << 23) && peak < 0x40000000ull &&
                       fits_costs32(n, 2 * (top + (peak >> K) + 1));
    uint64_t best = ~0ull;
    if (__builtin_expect(__all(small), 1)) {
      Costs32 acc;
      acc.clear();
      const int32_t h = (int32_t)half;
      auto zigzag_of = [&](int32_t x, int32_t y, int32_t z, int32_t v) {
        const int32_t s = __mul24(n0, x) + __mul24(n1, y) + __mul24(n2, z) + h;
        const int32_t r = v - (s >> K);
        return (uint32_t)((r << 1) ^ (r >> 31));
      };
      auto zigzag = [&](uint32_t i) { return zigzag_of(a0[i], b0[i], c0[i], v0[i]); };
      const uint32_t cnt = (uint32_t)n;
      if constexpr (SL == 1 && MB == 1) {
        // the samples are the same in every lane: scalar loads, four samples
        // ahead
        uint32_t i = 0;
        if (cnt >= 4) {
          int32_t s0[4], s1[4], s2[4], s3[4];
          auto load = [&](uint32_t at) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              s0[q] = a0[at + q];
              s1[q] = b0[at + q];
              s2[q] = c0[at + q];
              s3[q] = v0[at + q];
            }
          };
          load(0);
          for (; i + 4 <= cnt; i += 4) {
            uint32_t u[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) u[q] = zigzag_of(s0[q], s1[q], s2[q], s3[q]);
            load(i + 8 <= cnt ? i + 4 : 0);
            acc.add2(u[0], u[1]);
            acc.add2(u[2], u[3]);
          }
        }
        for (; i < cnt; i += 2) {
          const uint32_t u0 = zigzag(i);
          acc.add2(u0, i + 1 < cnt ? zigzag(i + 1) : 0u);
        }
      } else {
        for (uint32_t i = slice; i < cnt; i += 2 * SL) {
          const bool two = i + SL < cnt;
          const uint32_t u = zigzag(i), v = zigzag(two ? i + SL : i);
          acc.add2(u, two ? v : 0u);
        }
      }
      acc.totals(n, [](auto v) { return group_sum<CB, G>(v); },
                 [&](int, uint64_t t) { best = t < best ? t : best; });
    } else {
      // Codes past 23 bits.  Many candidates: every coder in one pass over the
      // samples, leading zeros counted in 32 bits (60 candidates on 4,000
      // meshlets 119 us, 33 on 20,000 478; five passes of four coders 402 and
      // 1,690).  Few, or more than 2^25 samples: four coders a pass, whose
      // registers leave the path above its waves (1 on 20,000 meshlets 63 us).
      auto value = [&](int32_t x, int32_t y, int32_t z, int32_t v) {
        const int64_t s = (int64_t)n0 * x + (int64_t)n1 * y + (int64_t)n2 * z;
        return zz64((int64_t)v - (K ? ((s + half) >> K) : s));
      };
      auto take = [&](int j, uint64_t acc) {
        const uint64_t t = body_bits(j, coder_sum(j, group_sum<CB, G>(acc), n), n);
        best = t < best ? t : best;
      };
      if (CB >= 16 && __all(n < (1u << 25))) {
        uint64_t rice[kRiceK];
        uint32_t zeros[kEgK];
#pragma unroll
        for (int k = 0; k < kRiceK; ++k) rice[k] = 0;
#pragma unroll
        for (int k = 0; k < kEgK; ++k) zeros[k] = 0;
        auto add = [&](uint64_t u) {
#pragma unroll
          for (int k = 0; k < kRiceK; ++k) rice[k] += u >> k;
#pragma unroll
          for (int k = 0; k < kEgK; ++k) zeros[k] += (uint32_t)__builtin_clzll(u + (1ull << k));
        };
        const uint32_t cnt = (uint32_t)n;
        uint32_t i = slice;
        for (; i + SL < cnt; i += 2 * SL) {   // two samples' loads a trip
          const int32_t x0 = a0[i], y0 = b0[i], z0 = c0[i], w0 = v0[i];
          const int32_t x1 = a0[i + SL], y1 = b0[i + SL], z1 = c0[i + SL], w1 = v0[i + SL];
          add(value(x0, y0, z0, w0));
          add(value(x1, y1, z1, w1));
        }
        if (i < cnt) add(value(a0[i], b0[i], c0[i], v0[i]));
#pragma unroll
        for (int k = 0; k < kRiceK; ++k) take(k, rice[k]);
#pragma unroll
        for (int k = 0; k < kEgK; ++k) take(kRiceK + k, zeros[k]);
      } else {
#pragma unroll 1
        for (int j0 = 0; j0 < kCoders; j0 += 4) {
          uint64_t acc[4] = {0, 0, 0, 0};
          for (uint64_t i = slice; i < n; i += SL) {
            const uint64_t u = value(a0[i], b0[i], c0[i], v0[i]);
#pragma unroll
            for (int q = 0; q < 4; ++q)
              acc[q] += j0 < kRiceK ? u >> (j0 + q)
                                    : (uint32_t)__builtin_clzll(u + (1ull << (j0 + q - kRiceK)));
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) take(j0 + q, acc[q]);
        }
      }
    }
    if (per_m) {
      if (slice == 0 && m < n_m && sc < S) per_m[m * S + sc] = (int64_t)best;
    } else {
      sum += best;
    }
  }
  if (per_m) return;
  part[wave][lane] = slice == 0 ? sum : 0ull;
  __syncthreads();
  if (threadIdx.x < CB && sc < S) {
    unsigned long long t = 0;
    for (int w = 0; w < kIrlpWaves; ++w)
      for (int q = 0; q < MB; ++q) t += part[w][q * G + c];
    atomicAdd(&cost[sc], t);
  }
}

// Waves that fill the chip's SIMDs several times over; more would only add
// atomics.
constexpr int64_t kIrlpGrid = 1024;

static hipError_t launch_irlp(const int32_t* a, const int32_t* b, const int32_t* c, const int32_t* v,
                              const int64_t* off, int64_t n_m, const int32_t* cand, int S, int K,
                              unsigned long long* cost, int64_t* per_m, hipStream_t st) {
#define IRLP(CB, SL, MB)                                                                        \
  do {                                                                                          \
    const int64_t per = (int64_t)kIrlpWaves * MB;                                               \
    const int64_t blocks = (n_m + per - 1) / per;                                               \
    hipLaunchKernelGGL((irlp_cost_kernel<CB, SL, MB>),                                          \
                       dim3((unsigned)(blocks < kIrlpGrid ? blocks : kIrlpGrid),                \
                            (unsigned)((S + CB - 1) / CB)),                                     \
                       dim3(64 * kIrlpWaves), 0, st, a, b, c, v, off, n_m, cand, S, K, cost,    \
                       per_m);                                                                  \
  } while (0)
  if (S <= 1) IRLP(1, 16, 4);
  else if (S <= 2) IRLP(2, 16, 2);
  else if (S <= 4) IRLP(4, 16, 1);
  else if (S <= 8) IRLP(8, 8, 1);
  else if (S <= 16) IRLP(16, 4, 1);
  else if (S <= 32 && n_m >= kIrlpGrid) IRLP(32, 2, 1);
  else if (n_m >= kIrlpGrid) IRLP(64, 1, 1);
  // few meshlets, fewer waves than SIMDs: more, shorter waves (16 candidates on a quarter of the
  // samples each): 298 meshlets and 60 candidates 11 us, a wave a meshlet 21 us.
  // On 4,000 meshlets the quarters take 75 us, whole waves 66.
  else IRLP(16, 4, 1);
#undef IRLP
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The L1 fit behind a fit's seeds (_fit_irls, encoder/_irlp_fit.py:239-257):
// least squares, then up to kIrlsIters rounds with weights 1 / max(|r|, 1)
// until the weights of the fit move by less than 1e-6.  One launch a round,
// none waits for the host: every workgroup of round k sums the partial sums
// of round k - 1, solves the 3 x 3 system and goes on with its share of the
// samples; once a round has converged the rest pass its result on.  Bound by
// the launches (about 5 us each); on the host, an SVD a round, it was 21 of
// the 31 ms that encoding 65,536 triangles took.
//
// The unknowns are those of (a - c, b - c, c): the codes of a triangle differ
// by far less than their size, so a, b and c are nearly parallel columns,
// while these, scaled to unit length, are not, and the normal equations lose
// next to nothing in float64: over spheres, tori and heightfields of 1,000 to
// 65,536 triangles at 12 and 16 bits the weights are off by at most 1e-14
// (the SVD of a, b, c: 8e-14).  Where they are nearly parallel all the same (a
// pivot under 1e-6), or lengths differ by more than 1e7, the fit is left to
// the caller (flag 2).
// ---------------------------------------------------------------------------
constexpr int kIrlsIters = 12, kIrlsSums = 9, kIrlsMaxBlocks = 256;

struct IrlsState {
  double x[3];   // weights of (a - c, b - c, c)
  double flag;   // 0 going on, 1 converged, 2 left to the caller
};

__device__ __forceinline__ IrlsState irls_solve(const double (&s)[kIrlsSums]) {
  // s: pp pq pc qq qc cc, py qy cy
  IrlsState r{{0.0, 0.0, 0.0}, 2.0};
  if (!(s[0] > 0.0 && s[3] > 0.0 && s[5] > 0.0)) return r;
  if (!(s[0] > 1e-14 * s[5] && s[3] > 1e-14 * s[5])) return r;
  const double ip = 1.0 / sqrt(s[0]), iq = 1.0 / sqrt(s[3]), ic = 1.0 / sqrt(s[5]);
  const double l21 = s[1] * ip * iq, l31 = s[2] * ip * ic, g32 = s[4] * iq * ic;
  const double d2 = 1.0 - l21 * l21;
  if (!(d2 >= 1e-6)) return r;
  const double l22 = sqrt(d2), l32 = (g32 - l31 * l21) / l22;
  const double d3 = 1.0 - l31 * l31 - l32 * l32;
  if (!(d3 >= 1e-6)) return r;
  const double l33 = sqrt(d3);
  const double y1 = s[6] * ip, y2 = (s[7] * iq - l21 * y1) / l22,
               y3 = (s[8] * ic - l31 * y1 - l32 * y2) / l33;
  const double z3 = y3 / l33, z2 = (y2 - l32 * z3) / l22, z1 = y1 - l21 * z2 - l31 * z3;
  r.x[0] = z1 * ip;
  r.x[1] = z2 * iq;
  r.x[2] = z3 * ic;
  r.flag = 0.0;
  return r;
}

// ws: partial sums of even and odd rounds (blocks x 9 each), then the states.
// round k < kIrlsIters + 1 adds up its sums; the one after it only writes the
// result: out = w0, w1, w2 of (a, b, c), flag.
__global__ __launch_bounds__(256) void irls_kernel(const int32_t* __restrict__ A,
                                                   const int32_t* __restrict__ B,
                                                   const int32_t* __restrict__ C,
                                                   const int32_t* __restrict__ Vv, int64_t n, int k,
                                                   double* __restrict__ ws,
                                                   double* __restrict__ out) {
  __shared__ double sh[4][kIrlsSums];
  __shared__ IrlsState cur;
  const int tid = threadIdx.x, lane = tid & 63, blocks = gridDim.x;
  const double* prev = ws + (size_t)((k + 1) & 1) * kIrlsMaxBlocks * kIrlsSums;
  double* mine = ws + (size_t)(k & 1) * kIrlsMaxBlocks * kIrlsSums;
  IrlsState* states = reinterpret_cast<IrlsState*>(ws + 2 * kIrlsMaxBlocks * kIrlsSums);
  auto wave_sum_f64 = [](double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
  };
  if (k > 0) {
    if (tid < 64) {
      double s[kIrlsSums];
#pragma unroll
      for (int j = 0; j < kIrlsSums; ++j) {
        s[j] = 0.0;
        for (int q = lane; q < blocks; q += 64) s[j] += prev[q * kIrlsSums + j];
        s[j] = wave_sum_f64(s[j]);
      }
      if (lane == 0) {
        IrlsState r;
        IrlsState last{{0.0, 0.0, 0.0}, 0.0};
        if (k > 1) last = states[k - 2];
        if (last.flag != 0.0) {
          r = last;
        } else {
          r = irls_solve(s);
          if (r.flag == 0.0 && k > 1) {
            const double m0 = fabs(r.x[0] - last.x[0]), m1 = fabs(r.x[1] - last.x[1]);
            const double m2 = fabs((r.x[2] - r.x[0] - r.x[1]) - (last.x[2] - last.x[0] - last.x[1]));
            if (fmax(m0, fmax(m1, m2)) < 1e-6) r.flag = 1.0;
          }
        }
        cur = r;
        if (blockIdx.x == 0) {
          states[k - 1] = r;
          if (k == kIrlsIters + 1) {
            out[0] = r.x[0];
            out[1] = r.x[1];
            out[2] = r.x[2] - r.x[0] - r.x[1];
            out[3] = r.flag;
          }
        }
      }
    }
    __syncthreads();
    if (k == kIrlsIters + 1 || cur.flag != 0.0) return;
  }
  double s[kIrlsSums];
#pragma unroll
  for (int j = 0; j < kIrlsSums; ++j) s[j] = 0.0;
  const double x0 = k ? cur.x[0] : 0.0, x1 = k ? cur.x[1] : 0.0, x2 = k ? cur.x[2] : 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + tid; i < n; i += (int64_t)blocks * 256) {
    const int32_t ci = C[i];
    const double c = ci, p = (double)A[i] - c, q = (double)B[i] - c, y = Vv[i];
    double t = 1.0;
    if (k) t = 1.0 / fmax(fabs(y - (x0 * p + x1 * q + x2 * c)), 1.0);
    const double tp = t * p, tq = t * q, tc = t * c;
    s[0] += tp * p;
    s[1] += tp * q;
    s[2] += tp * c;
    s[3] += tq * q;
    s[4] += tq * c;
    s[5] += tc * c;
    s[6] += tp * y;
    s[7] += tq * y;
    s[8] += tc * y;
  }
#pragma unroll
  for (int j = 0; j < kIrlsSums; ++j) {
    const double v = wave_sum_f64(s[j]);
    if (lane == 0) sh[tid >> 6][j] = v;
  }
  __syncthreads();
  if (tid < kIrlsSums)
    mine[blockIdx.x * kIrlsSums + tid] = (sh[0][tid] + sh[1][tid]) + (sh[2][tid] + sh[3][tid]);
}

__global__ void zero_i64_kernel(int64_t* p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace stride

using namespace stride;

extern "C" int stride_stream_costs(const int32_t* d_vals, const int64_t* d_off, int64_t n_streams,
                                   int64_t* d_costs, void* stream) {
  if (n_streams < 0 || (n_streams && (!d_vals || !d_off || !d_costs)))
    return set_error(STRIDE_E_ARG, "stride_stream_costs: null argument");
  if (n_streams == 0) return STRIDE_OK;
  const hipError_t e =
      launch_streams(d_vals, d_off, n_streams, d_costs, nullptr, nullptr, (hipStream_t)stream);
  if (e != hipSuccess) return set_error(STRIDE_E_HIP, hipGetErrorString(e));
  return STRIDE_OK;
}

extern "C" int stride_select_codes(const int32_t* d_vals, const int64_t* d_off, int64_t n_streams,
                                   uint8_t* d_tagk, int64_t* d_bits, void* stream) {
  if (n_streams < 0 || (n_streams && (!d_vals || !d_off || !d_tagk)))
    return set_error(STRIDE_E_ARG, "stride_select_codes: null argument");
  if (n_streams == 0) return STRIDE_OK;
  const hipError_t e =
      launch_streams(d_vals, d_off, n_streams, nullptr, d_tagk, d_bits, (hipStream_t)stream);
  if (e != hipSuccess) return set_error(STRIDE_E_HIP, hipGetErrorString(e));
  return STRIDE_OK;
}

extern "C" int stride_irlp_cost(const int32_t* d_a, const int32_t* d_b, const int32_t* d_c,
                                const int32_t* d_v, const int64_t* d_off, int64_t n_m,
                                const int32_t* d_cand, int32_t S, int32_t K, int64_t* d_cost,
                                void* stream) {
  if (n_m < 0 || S < 0 || K < 0 || K > 30 || !d_cost || (S && !d_cand) ||
      (n_m && (!d_a || !d_b || !d_c || !d_v || !d_off)))
    return set_error(STRIDE_E_ARG, "stride_irlp_cost: invalid argument");
  if (S == 0) return STRIDE_OK;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(zero_i64_kernel, dim3((S + 255) / 256), dim3(256), 0, st, d_cost, (int)S);
  if (n_m > 0) {
    if (n_m > 0x7FFFFFFF) return set_error(STRIDE_E_ARG, "stride_irlp_cost: too many meshlets");
    const hipError_t le = launch_irlp(d_a, d_b, d_c, d_v, d_off, n_m, d_cand, (int)S, (int)K,
                                      reinterpret_cast<unsigned long long*>(d_cost), nullptr, st);
    if (le != hipSuccess) return set_error(STRIDE_E_HIP, hipGetErrorString(le));
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(STRIDE_E_HIP, hipGetErrorString(e));
  return STRIDE_OK;
}

extern "C" int stride_irlp_cost_meshlets(const int32_t* d_a, const int32_t* d_b, const int32_t* d_c,
                                         const int32_t* d_v, const int64_t* d_off, int64_t n_m,
                                         const int32_t* d_cand, int32_t S, int32_t K,
                                         int64_t* d_cost_m, void* stream) {
  if (n_m < 0 || S < 0 || K < 0 || K > 30 || (S && !d_cand) ||
      (n_m && (!d_a || !d_b || !d_c || !d_v || !d_off || !d_cost_m)))
    return set_error(STRIDE_E_ARG, "stride_irlp_cost_meshlets: invalid argument");
  if (S == 0 || n_m == 0) return STRIDE_OK;
  if (n_m > 0x7FFFFFFF) return set_error(STRIDE_E_ARG, "stride_irlp_cost_meshlets: too many meshlets");
  const hipError_t e = launch_irlp(d_a, d_b, d_c, d_v, d_off, n_m, d_cand, (int)S, (int)K, nullptr,
                                   d_cost_m, (hipStream_t)stream);
  if (e != hipSuccess) return set_error(STRIDE_E_HIP, hipGetErrorString(e));
  return STRIDE_OK;
}

extern "C" int stride_irls_ws_doubles(int64_t* doubles) {
  if (!doubles) return set_error(STRIDE_E_ARG, "stride_irls_ws_doubles: null argument");
  *doubles = 2 * kIrlsMaxBlocks * kIrlsSums + 4 * (kIrlsIters + 1);
  return STRIDE_OK;
}

extern "C" int stride_irls_fit(const int32_t* d_a, const int32_t* d_b, const int32_t* d_c,
                               const int32_t* d_v, int64_t n, double* d_ws, double* d_out,
                               void* stream) {
  if (n < 0 || !d_ws || !d_out || (n && (!d_a || !d_b || !d_c || !d_v)))
    return set_error(STRIDE_E_ARG, "stride_irls_fit: invalid argument");
  // at least two samples a thread, so that a workgroup's sums are worth its solve
  int64_t blocks = (n + 511) / 512;
  blocks = blocks < 1 ? 1 : (blocks > kIrlsMaxBlocks ? kIrlsMaxBlocks : blocks);
  for (int k = 0; k <= kIrlsIters + 1; ++k)
    hipLaunchKernelGGL(irls_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, d_a,
                       d_b, d_c, d_v, n, k, d_ws, d_out);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(STRIDE_E_HIP, hipGetErrorString(e));
  return STRIDE_OK;
}
