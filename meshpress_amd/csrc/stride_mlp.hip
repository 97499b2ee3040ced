// Learned coder/predictor proposal: a 32 -> 128 -> 128 -> 176 MLP with
// BF16 weights and activations and FP32 accumulation on the gfx950 matrix
// cores (v_mfma_f32_16x16x32_bf16), plus its backward pass, a grouped
// softmax cross-entropy and an Adam step.
//
// Parameter layout (float32 master copy, n_params = 43,440):
//   W1 32 x 128 | W2 128 x 128 | W3 128 x 176 | b1 128 | b2 128 | b3 176
// (W row-major, input index major).  The first 43,008 entries (the
// weights) also exist as a bf16 copy that the GEMMs read.
//
// Output heads (logit columns): three predictor heads of 17 classes (one
// per axis, columns 0..50) and six coder heads of 20 classes (one per
// residual stream dx dy dz px py pz, columns 51..170); columns 171..175 pad
// the width to a multiple of 16 and never enter a softmax.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <type_traits>

#include "../../include/stride_hip.h"
#include "stride_err.h"

namespace stride {
namespace mlp {

constexpr int kIn = 32, kHid = 128, kOut = 176;
constexpr int kHeads = 9;
constexpr int kNW = kIn * kHid + kHid * kHid + kHid * kOut;   // 43,008
constexpr int kNP = kNW + kHid + kHid + kOut;                 // 43,440
__constant__ int kHeadOff[kHeads + 1] = {0, 17, 34, 51, 71, 91, 111, 131, 151, 171};

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// float -> bf16, round to nearest even (NaN stays a quiet NaN)
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

enum Epi : int { kEpiF32 = 0, kEpiBiasReluBf16 = 1, kEpiMaskBf16 = 2 };

struct GemmArgs {
  const uint16_t* A;   // op(A)[m][k] = transA ? A[k * lda + m] : A[m * lda + k]
  const uint16_t* B;   // op(B)[k][n] = transB ? B[n * ldb + k] : B[k * ldb + n]
  int lda, ldb, transA, transB;
  int M, N, K;
  int epi;
  const float* bias;     // N floats or null (kEpiF32, kEpiBiasReluBf16)
  const uint16_t* mask;  // kEpiMaskBf16: keep C[m][n] where mask[m * ldm + n] > 0
  int ldm;
  float* Cf;             // kEpiF32 output
  uint16_t* Cb;          // bf16 outputs
  int ldc;
};

// C = op(A) op(B): a 256-thread workgroup owns a 64 x 64 tile of C; wave w
// owns rows 16w..16w+15 as four 16 x 16 MFMA tiles.  Each K step of 32
// stages the 64 x 32 slice of op(A) and the 32 x 64 slice of op(B) in LDS
// (zero outside the matrices), then every lane feeds its fragments of the
// gfx950 16 x 16 x 32 bf16 MFMA, eight k values each:
//   A: row = lane % 16, k = 8 (lane / 16) + i
//   B: col = lane % 16, k = 8 (lane / 16) + i
//   D: row = 4 (lane / 16) + i, col = lane % 16
__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs g) {
  __shared__ uint16_t As[64][32 + 4];
  __shared__ uint16_t Bs[32][64 + 4];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  f4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < g.K; k0 += 32) {
    // stage: 2048 elements of each operand, 8 per thread
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int e = t + 256 * r;
      {  // A slice: row e / 32, col e % 32
        const int mm = e >> 5, kk = e & 31;
        const int gm = m0 + mm, gk = k0 + kk;
        uint16_t v = 0;
        if (gm < g.M && gk < g.K)
          v = g.transA ? g.A[(size_t)gk * g.lda + gm] : g.A[(size_t)gm * g.lda + gk];
        As[mm][kk] = v;
      }
      {  // B slice: row e / 64, col e % 64
        const int kk = e >> 6, nn = e & 63;
        const int gk = k0 + kk, gn = n0 + nn;
        uint16_t v = 0;
        if (gk < g.K && gn < g.N)
          v = g.transB ? g.B[(size_t)gn * g.ldb + gk] : g.B[(size_t)gk * g.ldb + gn];
        Bs[kk][nn] = v;
      }
    }
    __syncthreads();
    const int fr = lane & 15, fk = (lane >> 4) * 8;
    bf8 a;
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = __builtin_bit_cast(__bf16, As[16 * w + fr][fk + i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bf8 b;
#pragma unroll
      for (int i = 0; i < 8; ++i) b[i] = __builtin_bit_cast(__bf16, Bs[fk + i][16 * j + fr]);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[j], 0, 0, 0);
    }
    __syncthreads();
  }
  const int col_in = lane & 15, row_in = (lane >> 4) * 4;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + 16 * j + col_in;
    if (n >= g.N) continue;
    const float bn = g.bias ? g.bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + 16 * w + row_in + i;
      if (m >= g.M) continue;
      const float x = acc[j][i];
      if (g.epi == kEpiF32) {
        g.Cf[(size_t)m * g.ldc + n] = x + bn;
      } else if (g.epi == kEpiBiasReluBf16) {
        const float y = x + bn;
        g.Cb[(size_t)m * g.ldc + n] = f2bf(y > 0.f ? y : 0.f);
      } else {
        const bool keep = bf2f(g.mask[(size_t)m * g.ldm + n]) > 0.f;
        g.Cb[(size_t)m * g.ldc + n] = f2bf(keep ? x : 0.f);
      }
    }
  }
}

// Heads, one lane per (sample, head): a block stages kHeadRows rows of
// logits in LDS with coalesced loads (stride kOut + 1: the lanes of one head
// read down a column, 177 mod 64 banks apart) and hands them to kHeadRows x 9
// of its lanes.  Bound by the exponentials' latency and the 704 B a row; a
// lane per sample walking its row in memory (every load of a wave in 64
// different lines, 16 blocks at 4,096 rows) took 83 us for the cross-entropy
// of 4,096 rows and 69 us for the heads of 4,000; this form 9 and 7 us.
constexpr int kHeadRows = 28;   // 28 x 9 = 252 of 256 lanes
struct HeadTile {
  float z[kHeadRows][kOut + 1];
};

__device__ __forceinline__ void load_head_tile(HeadTile& T, const float* __restrict__ z,
                                               int64_t b0, int rows) {
  const float* src = z + b0 * kOut;
#pragma unroll 5
  for (int i = threadIdx.x; i < rows * kOut; i += 256) T.z[i / kOut][i % kOut] = src[i];
}

// Grouped softmax cross-entropy: per sample and head h with label y
// (255 = head ignored): loss += logsumexp(z_h) - z_h[y];
// dz_h = scale * (softmax(z_h) - onehot(y)), written as bf16.
__global__ __launch_bounds__(256) void xent_kernel(const float* __restrict__ z,
                                                   const uint8_t* __restrict__ labels, int64_t n,
                                                   float scale, uint16_t* __restrict__ dz,
                                                   float* __restrict__ loss) {
  __shared__ HeadTile T;
  __shared__ float Lh[kHeadRows][kHeads];
  const int64_t b0 = (int64_t)blockIdx.x * kHeadRows;
  const int rows = (int)(n - b0 < kHeadRows ? n - b0 : kHeadRows);
  const int r = threadIdx.x / kHeads, h = threadIdx.x % kHeads;
  load_head_tile(T, z, b0, rows);
  __syncthreads();
  if (r < rows) {
    const int o = kHeadOff[h], c = kHeadOff[h + 1] - o;
    float* zr = T.z[r];
    const int y = labels[(b0 + r) * kHeads + h];
    // the logits' places take the gradient
    if (y == 255 || y >= c) {
      for (int j = 0; j < c; ++j) zr[o + j] = 0.f;
      Lh[r][h] = 0.f;
    } else {
      float mx = zr[o];
      for (int j = 1; j < c; ++j) mx = fmaxf(mx, zr[o + j]);
      const float zy = zr[o + y];
      float s = 0.f;
      for (int j = 0; j < c; ++j) {
        const float e = expf(zr[o + j] - mx);
        s += e;
        zr[o + j] = e;
      }
      Lh[r][h] = logf(s) + mx - zy;
      const float inv = 1.f / s;
      for (int j = 0; j < c; ++j) {
        const float p = zr[o + j] * inv;
        zr[o + j] = scale * (p - (j == y ? 1.f : 0.f));
      }
    }
    if (h == 0)
      for (int j = kHeadOff[kHeads]; j < kOut; ++j) zr[j] = 0.f;
  }
  __syncthreads();
  uint16_t* out = dz + b0 * kOut;
#pragma unroll 5
  for (int i = threadIdx.x; i < rows * kOut; i += 256) out[i] = f2bf(T.z[i / kOut][i % kOut]);
  if (loss && threadIdx.x < (unsigned)rows) {
    float L = 0.f;
#pragma unroll
    for (int j = 0; j < kHeads; ++j) L += Lh[threadIdx.x][j];
    loss[b0 + threadIdx.x] = L;
  }
}

// Inference heads: predictor heads as probabilities (n x 51 float), coder
// heads as arg-max class (lowest index on ties) and its probability.
__global__ __launch_bounds__(256) void heads_kernel(const float* __restrict__ z, int64_t n,
                                                    float* __restrict__ pred_prob,
                                                    uint8_t* __restrict__ cls,
                                                    float* __restrict__ cls_prob) {
  __shared__ HeadTile T;
  constexpr int kPred = 51;
  const int64_t b0 = (int64_t)blockIdx.x * kHeadRows;
  const int rows = (int)(n - b0 < kHeadRows ? n - b0 : kHeadRows);
  const int r = threadIdx.x / kHeads, h = threadIdx.x % kHeads;
  load_head_tile(T, z, b0, rows);
  __syncthreads();
  if (r < rows) {
    const int o = kHeadOff[h], c = kHeadOff[h + 1] - o;
    float* zr = T.z[r];
    float mx = zr[o];
    int am = 0;
    for (int j = 1; j < c; ++j)
      if (zr[o + j] > mx) { mx = zr[o + j]; am = j; }
    float s = 0.f;
    for (int j = 0; j < c; ++j) {
      const float e = expf(zr[o + j] - mx);
      s += e;
      if (h < 3) zr[o + j] = e;
    }
    const float inv = 1.f / s;
    if (h < 3) {
      for (int j = 0; j < c; ++j) zr[o + j] *= inv;
    } else {
      cls[(b0 + r) * 6 + (h - 3)] = (uint8_t)am;
      cls_prob[(b0 + r) * 6 + (h - 3)] = inv;   // exp(0) / s
    }
  }
  __syncthreads();
  float* out = pred_prob + b0 * kPred;
  for (int i = threadIdx.x; i < rows * kPred; i += 256) out[i] = T.z[i / kPred][i % kPred];
}

// ---------------------------------------------------------------------------
// The network's own passes.  Every layer is small (86 KB of bf16 weights), so
// three launches of a tiled product spend their time in latencies; here a
// block keeps the weights of a whole pass in LDS (rows padded by 8: a
// fragment's 16 rows then start 16 bytes x 16 banks apart, so its 16-byte
// reads are conflict free) and takes tiles of 16 MT rows of the batch through
// every layer.  The matrix products take the fragments of gemm_kernel in its
// k order, so each output has gemm_kernel's bits.  Bound by latency: staging
// the weights (L2), then LDS reads between barriers.  4,096 rows: forward
// 12.3 us (three gemm_kernel launches: 42 us), hidden gradients 14.8 us,
// weight gradients and their sum 19.5 + 7 us.  gemm_kernel and a serial
// column sum took 4.0 ms for the backward pass: a product over the batch has
// 6 tiles of 64 x 64, so 6 of 256 CUs walked its 4,096 rows, and the column
// sums ran in one block.
// ---------------------------------------------------------------------------
constexpr int kLd1 = kIn + 8;          // rows of 32 k values
constexpr int kLd2 = kHid + 8;         // rows of 128
constexpr int kK3 = 192, kLd3 = kK3 + 8;   // 176 logits, zero to whole k steps of 32
constexpr int kMaxPassBlocks = 256;    // one block of a pass per CU (its LDS allows no more)

// eight consecutive bf16 values; ALIGNED: p is 16-byte aligned
template <bool ALIGNED>
__device__ __forceinline__ uint4 load8(const uint16_t* __restrict__ p) {
  if constexpr (ALIGNED) return *reinterpret_cast<const uint4*>(p);
  uint4 v;
  v.x = p[0] | ((uint32_t)p[1] << 16);
  v.y = p[2] | ((uint32_t)p[3] << 16);
  v.z = p[4] | ((uint32_t)p[5] << 16);
  v.w = p[6] | ((uint32_t)p[7] << 16);
  return v;
}
template <bool ALIGNED>
__device__ __forceinline__ void store8(uint16_t* __restrict__ p, uint4 v) {
  if constexpr (ALIGNED) {
    *reinterpret_cast<uint4*>(p) = v;
  } else {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[2 * i] = (uint16_t)w[i];
      p[2 * i + 1] = (uint16_t)(w[i] >> 16);
    }
  }
}
// fragment of a row-major LDS matrix: row `row`, k values k0 + 8 (lane / 16) + i
__device__ __forceinline__ bf8 frag(const uint16_t* m, int ld, int row, int k0, int lane) {
  return __builtin_bit_cast(bf8, *reinterpret_cast<const uint4*>(m + row * ld + k0 + 8 * (lane >> 4)));
}
__device__ __forceinline__ f4 mma(bf8 a, bf8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// rows r0.. of a row-major (n x C) matrix -> LDS rows of stride ld, zero past n
template <int C, int ROWS, bool ALIGNED>
__device__ __forceinline__ void load_rows(uint16_t* dst, int ld, const uint16_t* __restrict__ src,
                                          int64_t r0, int64_t n) {
  constexpr int oct = C / 8;
  for (int u = threadIdx.x; u < ROWS * oct; u += 256) {
    const int r = u / oct, c = u % oct;
    uint4 v{0u, 0u, 0u, 0u};
    if (r0 + r < n) v = load8<ALIGNED>(src + (r0 + r) * C + 8 * c);
    *reinterpret_cast<uint4*>(dst + r * ld + 8 * c) = v;
  }
}
template <int C, int ROWS, bool ALIGNED>
__device__ __forceinline__ void store_rows(uint16_t* __restrict__ dst, const uint16_t* src, int ld,
                                           int64_t r0, int64_t n) {
  constexpr int oct = C / 8;
  for (int u = threadIdx.x; u < ROWS * oct; u += 256) {
    const int r = u / oct, c = u % oct;
    if (r0 + r < n)
      store8<ALIGNED>(dst + (r0 + r) * C + 8 * c, *reinterpret_cast<const uint4*>(src + r * ld + 8 * c));
  }
}
// ROWS rows of C columns -> columns: dst[col * ld + row] (two rows a word)
template <int C, int ROWS, bool ALIGNED>
__device__ __forceinline__ void load_cols(uint16_t* dst, int ld, const uint16_t* __restrict__ src,
                                          int64_t r0, int64_t n) {
  constexpr int oct = C / 8;
  for (int u = threadIdx.x; u < (ROWS / 2) * oct; u += 256) {
    // eight row pairs of one octet are neighbouring lanes: their words fall
    // in neighbouring banks
    const int rp = (u & 7) + 8 * (u / (8 * oct)), c = (u >> 3) % oct;
    uint4 a{0u, 0u, 0u, 0u}, b{0u, 0u, 0u, 0u};
    if (r0 + 2 * rp < n) a = load8<ALIGNED>(src + (r0 + 2 * rp) * C + 8 * c);
    if (r0 + 2 * rp + 1 < n) b = load8<ALIGNED>(src + (r0 + 2 * rp + 1) * C + 8 * c);
    const uint32_t av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t* d = reinterpret_cast<uint32_t*>(dst + (8 * c + 2 * i) * ld + 2 * rp);
      d[0] = (av[i] & 0xFFFFu) | (bv[i] << 16);
      d[ld / 2] = (av[i] >> 16) | (bv[i] & 0xFFFF0000u);
    }
  }
}

template <int MT>
constexpr int forward_lds() {
  return 2 * (kHid * kLd1 + kHid * kLd2 + kOut * kLd2 + 16 * MT * (kLd1 + 2 * kLd2));
}

// One layer of the forward pass: column tiles w, w + 4, ... of the tile's
// rows; relu(A W + b) as bf16 into H.
template <int K, int MT>
__device__ __forceinline__ void hidden_layer(const uint16_t* A, int lda, const uint16_t* Wt, int ldw,
                                             const float* __restrict__ bias, uint16_t* H, int lane,
                                             int w) {
  const int fr = lane & 15, row_in = (lane >> 4) * 4;
#pragma unroll
  for (int j = w; j < kHid / 16; j += 4) {
    f4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 32) {
      const bf8 b = frag(Wt, ldw, 16 * j + fr, k0, lane);
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = mma(frag(A, lda, 16 * t + fr, k0, lane), b, acc[t]);
    }
    const float bn = bias[16 * j + fr];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float y = acc[t][i] + bn;
        H[(16 * t + row_in + i) * kLd2 + 16 * j + fr] = f2bf(y > 0.f ? y : 0.f);
      }
  }
}

template <int MT, bool ALIGNED>
__global__ __launch_bounds__(256) void forward_kernel(const uint16_t* __restrict__ x, int64_t n,
                                                      const uint16_t* __restrict__ wb,
                                                      const float* __restrict__ params,
                                                      uint16_t* __restrict__ h1,
                                                      uint16_t* __restrict__ h2,
                                                      float* __restrict__ z) {
  extern __shared__ uint4 lds[];
  uint16_t* W1t = reinterpret_cast<uint16_t*>(lds);
  uint16_t* W2t = W1t + kHid * kLd1;
  uint16_t* W3t = W2t + kHid * kLd2;
  uint16_t* X = W3t + kOut * kLd2;
  uint16_t* H1 = X + 16 * MT * kLd1;
  uint16_t* H2 = H1 + 16 * MT * kLd2;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int fr = lane & 15, row_in = (lane >> 4) * 4;
  const float *b1 = params + kNW, *b2 = b1 + kHid, *b3 = b2 + kHid;
  load_cols<kHid, kIn, ALIGNED>(W1t, kLd1, wb, 0, kIn);
  load_cols<kHid, kHid, ALIGNED>(W2t, kLd2, wb + kIn * kHid, 0, kHid);
  load_cols<kOut, kHid, ALIGNED>(W3t, kLd2, wb + kIn * kHid + kHid * kHid, 0, kHid);
  const int64_t tiles = (n + 16 * MT - 1) / (16 * MT);
  for (int64_t q = blockIdx.x; q < tiles; q += gridDim.x) {
    const int64_t r0 = q * 16 * MT;
    load_rows<kIn, 16 * MT, ALIGNED>(X, kLd1, x, r0, n);
    __syncthreads();
    hidden_layer<kIn, MT>(X, kLd1, W1t, kLd1, b1, H1, lane, w);
    __syncthreads();
    store_rows<kHid, 16 * MT, ALIGNED>(h1, H1, kLd2, r0, n);
    hidden_layer<kHid, MT>(H1, kLd2, W2t, kLd2, b2, H2, lane, w);
    __syncthreads();
    store_rows<kHid, 16 * MT, ALIGNED>(h2, H2, kLd2, r0, n);
    for (int j = w; j < kOut / 16; j += 4) {
      f4 acc[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k0 = 0; k0 < kHid; k0 += 32) {
        const bf8 b = frag(W3t, kLd2, 16 * j + fr, k0, lane);
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = mma(frag(H2, kLd2, 16 * t + fr, k0, lane), b, acc[t]);
      }
      const float bn = b3[16 * j + fr];
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int64_t m = r0 + 16 * t + row_in + i;
          if (m < n) z[m * kOut + 16 * j + fr] = acc[t][i] + bn;
        }
    }
  }
}

template <int MT>
constexpr int hidden_grad_lds() {
  return 2 * (kHid * kLd3 + kHid * kLd2 + 16 * MT * (kLd3 + 3 * kLd2));
}

// dH2 = (dZ W3^T) * (H2 > 0), dH1 = (dH2 W2^T) * (H1 > 0).  The weights'
// rows already run along k here.
template <int MT, bool ALIGNED>
__global__ __launch_bounds__(256) void hidden_grad_kernel(const uint16_t* __restrict__ dz, int64_t n,
                                                          const uint16_t* __restrict__ wb,
                                                          const uint16_t* __restrict__ h1,
                                                          const uint16_t* __restrict__ h2,
                                                          uint16_t* __restrict__ dh2,
                                                          uint16_t* __restrict__ dh1) {
  extern __shared__ uint4 lds[];
  uint16_t* W3 = reinterpret_cast<uint16_t*>(lds);
  uint16_t* W2 = W3 + kHid * kLd3;
  uint16_t* Z = W2 + kHid * kLd2;
  uint16_t* M2 = Z + 16 * MT * kLd3;   // H2, then dH1
  uint16_t* M1 = M2 + 16 * MT * kLd2;
  uint16_t* D2 = M1 + 16 * MT * kLd2;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int fr = lane & 15, row_in = (lane >> 4) * 4;
  load_rows<kOut, kHid, ALIGNED>(W3, kLd3, wb + kIn * kHid + kHid * kHid, 0, kHid);
  load_rows<kHid, kHid, ALIGNED>(W2, kLd2, wb + kIn * kHid, 0, kHid);
  const uint4 zero{0u, 0u, 0u, 0u};
  for (int u = threadIdx.x; u < 2 * kHid; u += 256)
    *reinterpret_cast<uint4*>(W3 + (u >> 1) * kLd3 + kOut + 8 * (u & 1)) = zero;
  for (int u = threadIdx.x; u < 2 * 16 * MT; u += 256)
    *reinterpret_cast<uint4*>(Z + (u >> 1) * kLd3 + kOut + 8 * (u & 1)) = zero;
  const int64_t tiles = (n + 16 * MT - 1) / (16 * MT);
  for (int64_t q = blockIdx.x; q < tiles; q += gridDim.x) {
    const int64_t r0 = q * 16 * MT;
    load_rows<kOut, 16 * MT, ALIGNED>(Z, kLd3, dz, r0, n);
    load_rows<kHid, 16 * MT, ALIGNED>(M2, kLd2, h2, r0, n);
    load_rows<kHid, 16 * MT, ALIGNED>(M1, kLd2, h1, r0, n);
    __syncthreads();
    auto product = [&](auto kk, const uint16_t* A, int lda, const uint16_t* W, int ldw,
                       const uint16_t* mask, uint16_t* out) {
      constexpr int K = decltype(kk)::value;
#pragma unroll
      for (int j = w; j < kHid / 16; j += 4) {
        f4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k0 = 0; k0 < K; k0 += 32) {
          const bf8 b = frag(W, ldw, 16 * j + fr, k0, lane);
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[t] = mma(frag(A, lda, 16 * t + fr, k0, lane), b, acc[t]);
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int at = (16 * t + row_in + i) * kLd2 + 16 * j + fr;
            out[at] = f2bf(bf2f(mask[at]) > 0.f ? acc[t][i] : 0.f);
          }
      }
    };
    product(std::integral_constant<int, kK3>{}, Z, kLd3, W3, kLd3, M2, D2);
    __syncthreads();
    store_rows<kHid, 16 * MT, ALIGNED>(dh2, D2, kLd2, r0, n);
    product(std::integral_constant<int, kHid>{}, D2, kLd2, W2, kLd2, M1, M2);
    __syncthreads();
    store_rows<kHid, 16 * MT, ALIGNED>(dh1, M2, kLd2, r0, n);
    __syncthreads();   // M2 is read until here; the next tile loads it
  }
}

// Weight and bias gradients of one layer over one slice of the batch:
// A^T G (CA x CG) and G's column sums, as products over the slice's rows.
// Rows are staged as columns, 64 at a time; wave w owns the row tiles w,
// w + 4, ... of the output and every column tile.  The column sums are one
// more row tile whose A fragment is all ones (1.0 x g is exact), shared out
// over the waves.
constexpr int kSliceStage = 64, kLdS = kSliceStage + 8;

template <int CA, int CG, bool ALIGNED>
__device__ __forceinline__ void weight_grad(uint16_t* lds, const uint16_t* __restrict__ A,
                                            const uint16_t* __restrict__ G, int64_t r0, int64_t r1,
                                            float* __restrict__ gW, float* __restrict__ gb) {
  constexpr int MTA = CA / 16, NT = CG / 16, MW = (MTA + 3) / 4, BW = (NT + 3) / 4;
  uint16_t* At = lds;
  uint16_t* Gt = lds + CA * kLdS;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int fr = lane & 15, row_in = (lane >> 4) * 4;
  f4 acc[MW][NT], accb[BW];
#pragma unroll
  for (int t = 0; t < MW; ++t)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[t][j] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < BW; ++j) accb[j] = f4{0.f, 0.f, 0.f, 0.f};
  bf8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = __builtin_bit_cast(__bf16, (uint16_t)0x3F80);
  for (int64_t r = r0; r < r1; r += kSliceStage) {
    load_cols<CA, kSliceStage, ALIGNED>(At, kLdS, A, r, r1);
    load_cols<CG, kSliceStage, ALIGNED>(Gt, kLdS, G, r, r1);
    __syncthreads();
#pragma unroll
    for (int k0 = 0; k0 < kSliceStage; k0 += 32) {
      bf8 a[MW];
#pragma unroll
      for (int t = 0; t < MW; ++t)
        a[t] = frag(At, kLdS, 16 * ((w + 4 * t) % MTA) + fr, k0, lane);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const bf8 b = frag(Gt, kLdS, 16 * j + fr, k0, lane);
#pragma unroll
        for (int t = 0; t < MW; ++t)
          if (w + 4 * t < MTA) acc[t][j] = mma(a[t], b, acc[t][j]);
        if (j % 4 == w) accb[j / 4] = mma(ones, b, accb[j / 4]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < MW; ++t)
    if (w + 4 * t < MTA)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          gW[(16 * (w + 4 * t) + row_in + i) * CG + 16 * j + fr] = acc[t][j][i];
  if (row_in == 0)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (j % 4 == w) gb[16 * j + fr] = accb[j / 4][0];
}

constexpr int kWeightGradLds = 2 * (kHid + kOut) * kLdS;

// blockIdx.y = layer (0: the output layer, the most work, first), blockIdx.x
// = slice of `slice` rows.  Slice i writes its gradient to out + i kNP.
template <bool ALIGNED>
__global__ __launch_bounds__(256) void weight_grad_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ h1,
    const uint16_t* __restrict__ h2, const uint16_t* __restrict__ dh1,
    const uint16_t* __restrict__ dh2, const uint16_t* __restrict__ dz, int64_t n, int64_t slice,
    float* __restrict__ out) {
  extern __shared__ uint4 lds4[];
  uint16_t* lds = reinterpret_cast<uint16_t*>(lds4);
  const int64_t r0 = blockIdx.x * slice, r1 = r0 + slice < n ? r0 + slice : n;
  float* g = out + (size_t)blockIdx.x * kNP;
  float* gb = g + kNW;
  if (blockIdx.y == 0)
    weight_grad<kHid, kOut, ALIGNED>(lds, h2, dz, r0, r1, g + kIn * kHid + kHid * kHid, gb + 2 * kHid);
  else if (blockIdx.y == 1)
    weight_grad<kHid, kHid, ALIGNED>(lds, h1, dh2, r0, r1, g + kIn * kHid, gb + kHid);
  else
    weight_grad<kIn, kHid, ALIGNED>(lds, x, dh1, r0, r1, g, gb);
}

// grad = sum of the slices' gradients, in slice order
__global__ __launch_bounds__(256) void sum_slices_kernel(const float* __restrict__ part, int slices,
                                                         float* __restrict__ grad) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kNP) return;
  float s = part[i];
#pragma unroll 8
  for (int q = 1; q < slices; ++q) s += part[(size_t)q * kNP + i];
  grad[i] = s;
}

// Adam (Kingma & Ba 2015) with bias correction folded into c1 = 1/(1-b1^t),
// c2 = 1/(1-b2^t); refreshes the bf16 copy of the weights.
__global__ __launch_bounds__(256) void adam_kernel(float* __restrict__ p, float* __restrict__ m,
                                                   float* __restrict__ v,
                                                   const float* __restrict__ g,
                                                   uint16_t* __restrict__ wb, int64_t n, int64_t n_w,
                                                   float lr, float b1, float b2, float eps,
                                                   float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  p[i] = pi;
  if (i < n_w) wb[i] = f2bf(pi);
}

__global__ __launch_bounds__(256) void to_bf16_kernel(const float* __restrict__ x, int64_t n,
                                                      uint16_t* __restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

static int launch_gemm(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.N <= 0 || g.K < 0) return set_error(STRIDE_E_ARG, "gemm: bad shape");
  const unsigned gx = (unsigned)((g.N + 63) / 64), gy = (unsigned)((g.M + 63) / 64);
  if ((g.M + 63) / 64 > 0x7FFFFFFF) return set_error(STRIDE_E_ARG, "gemm: M too large");
  hipLaunchKernelGGL(gemm_kernel, dim3(gx, gy), dim3(256), 0, st, g);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? STRIDE_OK : set_error(STRIDE_E_HIP, hipGetErrorString(e));
}

static GemmArgs gemm(const uint16_t* A, int lda, int tA, const uint16_t* B, int ldb, int tB, int M,
                     int N, int K, int epi, const float* bias, const uint16_t* mask, int ldm,
                     float* Cf, uint16_t* Cb, int ldc) {
  GemmArgs g;
  g.A = A; g.B = B; g.lda = lda; g.ldb = ldb; g.transA = tA; g.transB = tB;
  g.M = M; g.N = N; g.K = K; g.epi = epi; g.bias = bias; g.mask = mask; g.ldm = ldm;
  g.Cf = Cf; g.Cb = Cb; g.ldc = ldc;
  return g;
}

static int last(void) {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? STRIDE_OK : set_error(STRIDE_E_HIP, hipGetErrorString(e));
}

static bool aligned16(const void* a, const void* b, const void* c, const void* d) {
  return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d) & 15) == 0;
}

// Rows a block takes at once: 16, or 16 kWideTile once that still gives
// every CU a tile (65,536 rows: forward 50 us; 16-row tiles would read the
// weights' fragments from LDS four times as often).
constexpr int kWideTile = 4;
static bool wide_tiles(int64_t n) { return n >= 16 * kWideTile * (int64_t)kMaxPassBlocks; }
static dim3 pass_grid(int64_t n, int mt) {
  return dim3((unsigned)std::min<int64_t>((n + 16 * mt - 1) / (16 * mt), kMaxPassBlocks));
}
// Slices of the weight gradients: one per kSliceStage rows, 64 at most (64
// slices of three layers fill 192 CUs, and each slice costs a 174 KB partial
// gradient written and read).
static int grad_slices(int64_t n) {
  return (int)std::min<int64_t>((n + kSliceStage - 1) / kSliceStage, 64);
}

}  // namespace mlp
}  // namespace stride

using namespace stride::mlp;
using stride::set_error;

#define MLP_TRY(x)              \
  do {                          \
    int rc_ = (x);              \
    if (rc_ != STRIDE_OK) return rc_; \
  } while (0)

extern "C" {

int stride_mlp_sizes(int32_t* n_in, int32_t* n_hidden, int32_t* n_out, int32_t* n_weights,
                     int32_t* n_params) {
  if (n_in) *n_in = kIn;
  if (n_hidden) *n_hidden = kHid;
  if (n_out) *n_out = kOut;
  if (n_weights) *n_weights = kNW;
  if (n_params) *n_params = kNP;
  return STRIDE_OK;
}

int stride_mlp_gemm(const uint16_t* d_a, int32_t lda, int32_t trans_a, const uint16_t* d_b,
                    int32_t ldb, int32_t trans_b, int32_t M, int32_t N, int32_t K, int32_t epi,
                    const float* d_bias, const uint16_t* d_mask, int32_t ldm, float* d_cf,
                    uint16_t* d_cb, int32_t ldc, void* stream) {
  if (!d_a || !d_b || M <= 0 || N <= 0 || K <= 0 || epi < 0 || epi > 2 ||
      (epi == kEpiF32 && !d_cf) || (epi != kEpiF32 && !d_cb) || (epi == kEpiMaskBf16 && !d_mask) ||
      lda <= 0 || ldb <= 0 || ldc < N)
    return set_error(STRIDE_E_ARG, "stride_mlp_gemm: invalid argument");
  if ((trans_a ? lda < M : lda < K) || (trans_b ? ldb < K : ldb < N) ||
      (epi == kEpiMaskBf16 && ldm < N))
    return set_error(STRIDE_E_ARG, "stride_mlp_gemm: leading dimension too small");
  return launch_gemm(gemm(d_a, lda, trans_a, d_b, ldb, trans_b, M, N, K, epi, d_bias, d_mask, ldm,
                          d_cf, d_cb, ldc),
                     (hipStream_t)stream);
}

int stride_mlp_forward(const uint16_t* d_x, int64_t n, const uint16_t* d_wb, const float* d_params,
                       uint16_t* d_h1, uint16_t* d_h2, float* d_z, void* stream) {
  if (n <= 0 || n > 0x7FFFFFFF || !d_x || !d_wb || !d_params || !d_h1 || !d_h2 || !d_z)
    return set_error(STRIDE_E_ARG, "stride_mlp_forward: invalid argument");
  hipStream_t st = (hipStream_t)stream;
  const bool al = aligned16(d_x, d_wb, d_h1, d_h2);
#define MLP_FORWARD(MT, AL)                                                                     \
  hipLaunchKernelGGL((forward_kernel<MT, AL>), pass_grid(n, MT), dim3(256), forward_lds<MT>(), st, \
                     d_x, n, d_wb, d_params, d_h1, d_h2, d_z)
  if (wide_tiles(n)) {
    if (al) MLP_FORWARD(kWideTile, true); else MLP_FORWARD(kWideTile, false);
  } else {
    if (al) MLP_FORWARD(1, true); else MLP_FORWARD(1, false);
  }
#undef MLP_FORWARD
  return last();
}

int stride_mlp_xent(const float* d_z, const uint8_t* d_labels, int64_t n, float scale,
                    uint16_t* d_dz, float* d_loss, void* stream) {
  if (n <= 0 || !d_z || !d_labels || !d_dz) return set_error(STRIDE_E_ARG, "stride_mlp_xent: invalid argument");
  hipLaunchKernelGGL(xent_kernel, dim3((unsigned)((n + kHeadRows - 1) / kHeadRows)), dim3(256), 0,
                     (hipStream_t)stream, d_z, d_labels, n, scale, d_dz, d_loss);
  return last();
}

int stride_mlp_backward_ws_floats(int64_t n, int64_t* floats) {
  if (n <= 0 || !floats)
    return set_error(STRIDE_E_ARG, "stride_mlp_backward_ws_floats: invalid argument");
  *floats = (int64_t)grad_slices(n) * kNP;
  return STRIDE_OK;
}

int stride_mlp_backward_ws(const uint16_t* d_x, int64_t n, const uint16_t* d_wb,
                           const uint16_t* d_h1, const uint16_t* d_h2, const uint16_t* d_dz,
                           uint16_t* d_dh2, uint16_t* d_dh1, float* d_grad, float* d_ws,
                           int64_t ws_floats, void* stream) {
  if (n <= 0 || n > 0x7FFFFFFF || !d_x || !d_wb || !d_h1 || !d_h2 || !d_dz || !d_dh2 || !d_dh1 ||
      !d_grad || ws_floats < 0 || (ws_floats && !d_ws))
    return set_error(STRIDE_E_ARG, "stride_mlp_backward: invalid argument");
  hipStream_t st = (hipStream_t)stream;
  const bool al = aligned16(d_x, d_wb, d_h1, d_h2) && aligned16(d_dz, d_dh2, d_dh1, d_dh1);
#define MLP_HIDDEN_GRAD(MT, AL)                                                                  \
  hipLaunchKernelGGL((hidden_grad_kernel<MT, AL>), pass_grid(n, MT), dim3(256),                  \
                     hidden_grad_lds<MT>(), st, d_dz, n, d_wb, d_h1, d_h2, d_dh2, d_dh1)
  if (wide_tiles(n)) {
    if (al) MLP_HIDDEN_GRAD(kWideTile, true); else MLP_HIDDEN_GRAD(kWideTile, false);
  } else {
    if (al) MLP_HIDDEN_GRAD(1, true); else MLP_HIDDEN_GRAD(1, false);
  }
#undef MLP_HIDDEN_GRAD
  MLP_TRY(last());
  // without room for the slices one block a layer takes the whole batch
  int slices = grad_slices(n);
  if (ws_floats < (int64_t)slices * kNP) slices = 1;
  const int64_t slice = ((n + slices - 1) / slices + kSliceStage - 1) / kSliceStage * kSliceStage;
  slices = (int)((n + slice - 1) / slice);
  float* out = slices > 1 ? d_ws : d_grad;
  hipLaunchKernelGGL(al ? weight_grad_kernel<true> : weight_grad_kernel<false>,
                     dim3((unsigned)slices, 3), dim3(256), kWeightGradLds, st, d_x, d_h1, d_h2,
                     d_dh1, d_dh2, d_dz, n, slice, out);
  MLP_TRY(last());
  if (slices == 1) return STRIDE_OK;
  hipLaunchKernelGGL(sum_slices_kernel, dim3((kNP + 255) / 256), dim3(256), 0, st, d_ws, slices,
                     d_grad);
  return last();
}

int stride_mlp_backward(const uint16_t* d_x, int64_t n, const uint16_t* d_wb, const uint16_t* d_h1,
                        const uint16_t* d_h2, const uint16_t* d_dz, uint16_t* d_dh2,
                        uint16_t* d_dh1, float* d_grad, void* stream) {
  return stride_mlp_backward_ws(d_x, n, d_wb, d_h1, d_h2, d_dz, d_dh2, d_dh1, d_grad, nullptr, 0,
                                stream);
}

int stride_mlp_adam(float* d_params, float* d_m, float* d_v, const float* d_grad, uint16_t* d_wb,
                    int64_t n_params, float lr, float beta1, float beta2, float eps, int32_t step,
                    void* stream) {
  if (!d_params || !d_m || !d_v || !d_grad || !d_wb || n_params != kNP || step < 1 ||
      !(beta1 >= 0.f && beta1 < 1.f) || !(beta2 >= 0.f && beta2 < 1.f) || !(eps > 0.f))
    return set_error(STRIDE_E_ARG, "stride_mlp_adam: invalid argument");
  const double p1 = std::pow((double)beta1, (double)step), p2 = std::pow((double)beta2, (double)step);
  const float c1 = (float)(1.0 / (1.0 - p1)), c2 = (float)(1.0 / (1.0 - p2));
  hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((n_params + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, d_params, d_m, d_v, d_grad, d_wb, n_params,
                     (int64_t)kNW, lr, beta1, beta2, eps, c1, c2);
  return last();
}

int stride_mlp_to_bf16(const float* d_x, int64_t n, uint16_t* d_y, void* stream) {
  if (n < 0 || (n && (!d_x || !d_y))) return set_error(STRIDE_E_ARG, "stride_mlp_to_bf16: invalid argument");
  if (n == 0) return STRIDE_OK;
  hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, d_x, n, d_y);
  return last();
}

int stride_mlp_heads(const float* d_z, int64_t n, float* d_pred_prob, uint8_t* d_cls,
                     float* d_cls_prob, void* stream) {
  if (n <= 0 || !d_z || !d_pred_prob || !d_cls || !d_cls_prob)
    return set_error(STRIDE_E_ARG, "stride_mlp_heads: invalid argument");
  hipLaunchKernelGGL(heads_kernel, dim3((unsigned)((n + kHeadRows - 1) / kHeadRows)), dim3(256), 0,
                     (hipStream_t)stream, d_z, n, d_pred_prob, d_cls, d_cls_prob);
  return last();
}

}  // extern "C"
