// mlp.hip — next-treelet predictor: BF16 MFMA MLP with FP32 accumulation.
//
// No counterpart in the reference, whose RT unit only has popularity
// heuristics (src/gpgpu-sim/shader.cc:3419-3559).  The model predicts, at a
// treelet transition of a ray, which treelet the ray enters next:
//   x  = [E[cur] (32) | one-hot octant of the ray direction (8) | depth/32 (1) |
//         E[h1] E[h2] E[h3] E[h4] (4 x 32)]           169 inputs, padded to 192
//   h1 = relu(x W1 + b1)       128
//   h2 = relu(h1 W2 + b2)      128
//   q  = h2 W3 + b3            32
//   logit[c] = q . O[c] + o[c] over the output classes (softmax, top-4)
// Every matrix product runs on v_mfma_f32_16x16x32_bf16: operands are rounded
// to BF16 (round to nearest even) as they are loaded, accumulation is FP32.
// Parameters are FP32 master copies updated with Adam.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "rtx.h"

namespace {

constexpr int kEmb = 32;
constexpr int kHid = 128;
constexpr int kIn = 169;
constexpr int kInPad = 192;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---- GEMM: C[M x N] (+)= op(A)[M x K] . op(B)[K x N], FP32 in memory --------
// 256 threads = 4 waves, each wave a 32x32 tile as 2x2 MFMA 16x16 tiles; the
// block tile is 64x64 (2x2 waves) or, for N <= 32, 128x32 (4x1 waves).
// MFMA 16x16x32 operand layout: lane l supplies row/column l % 16 and the 8
// consecutive k values starting at 8 * (l / 16); the result holds rows
// 4 * (l / 16) + i (i < 4) of column l % 16.  With gridDim.z > 1 the K range
// is split across blocks and the partial products are added into C atomically
// (C already holds the addend: zero or the value to accumulate into).
template <bool TA, bool TB, int BN>
__global__ __launch_bounds__(256) void gemm_bf16(int M, int N, int K, int k_chunk, const float* __restrict__ A,
                                                 int lda, const float* __restrict__ B, int ldb, float* __restrict__ C,
                                                 int ldc, int accumulate) {
  constexpr int WAVES_N = BN / 32;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int row0 = blockIdx.y * (128 / WAVES_N) + (wave / WAVES_N) * 32;
  const int col0 = blockIdx.x * BN + (wave % WAVES_N) * 32;
  const int r16 = lane & 15, kq = (lane >> 4) * 8;
  const int kb = blockIdx.z * k_chunk;
  const int ke = min(K, kb + k_chunk);
  f32x4 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = kb; k0 < ke; k0 += 32) {
    bf16x8 a[2], b[2];
    for (int i = 0; i < 2; ++i) {
      const int m = row0 + i * 16 + r16;
      for (int t = 0; t < 8; ++t) {
        const int k = k0 + kq + t;
        float v = 0.f;
        if (m < M && k < ke) v = TA ? A[(size_t)k * lda + m] : A[(size_t)m * lda + k];
        a[i][t] = (__bf16)v;
      }
    }
    for (int j = 0; j < 2; ++j) {
      const int n = col0 + j * 16 + r16;
      for (int t = 0; t < 8; ++t) {
        const int k = k0 + kq + t;
        float v = 0.f;
        if (n < N && k < ke) v = TB ? B[(size_t)n * ldb + k] : B[(size_t)k * ldb + n];
        b[j][t] = (__bf16)v;
      }
    }
    for (int i = 0; i < 2; ++i)
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
  }
  const bool split = gridDim.z > 1;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) {
      const int n = col0 + j * 16 + r16;
      for (int t = 0; t < 4; ++t) {
        const int m = row0 + i * 16 + (lane >> 4) * 4 + t;
        if (m < M && n < N) {
          float* c = C + (size_t)m * ldc + n;
          if (split)
            atomicAdd(c, acc[i][j][t]);
          else
            *c = accumulate ? *c + acc[i][j][t] : acc[i][j][t];
        }
      }
    }
}

__global__ void zero_rows(float* C, int M, int N, int ldc) {
  const size_t total = (size_t)M * N;
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < total; k += (size_t)gridDim.x * blockDim.x)
    C[(k / N) * ldc + k % N] = 0.f;
}

// ---- trunk: x -> h1 -> h2 -> q in one kernel ------------------------------------
// Matrices as MFMA operands: fragment (column tile ct, 32-deep step ks) of a
// K x N matrix holds, for lane l, the eight k values 32 ks + 8 (l / 16) + t of
// column 16 ct + l % 16, rounded to BF16, at [(ct * KS + ks) * 64 + l].  The
// forward pass takes W1, W2, W3, the backward pass their transposes.
constexpr int kFrag1 = 0;                                        // W1: 192 x 128
constexpr int kFrag2 = kFrag1 + (kHid / 16) * (kInPad / 32);     // W2: 128 x 128
constexpr int kFrag3 = kFrag2 + (kHid / 16) * (kHid / 32);       // W3: 128 x 32
constexpr int kFragForward = kFrag3 + (kEmb / 16) * (kHid / 32);
constexpr int kFragT3 = kFragForward;                            // W3^T: 32 x 128
constexpr int kFragT2 = kFragT3 + (kHid / 16) * (kEmb / 32);     // W2^T: 128 x 128
constexpr int kFragT1 = kFragT2 + (kHid / 16) * (kHid / 32);     // W1^T: 128 x 192
constexpr int kFragEnd = kFragT1 + (kInPad / 16) * (kHid / 32);
struct Weights {
  const float *W1, *b1, *W2, *b2, *W3, *b3;
};

// The tile row paired with k-slot 8g + j of an MFMA that takes a result tile as
// its operand (see the fused output layer).
__device__ __forceinline__ int kslot_row(int g, int j) { return j < 4 ? 4 * g + j : 16 + 4 * g + j - 4; }

// One wave per fragment: `count` of the trunk's, then (training) the output
// layer's: for each 16 classes the rows' fragment (lane: class c16, elements
// 8g..8g+7), for each 32 classes and half e of the embedding the columns'
// fragment (lane: element 16e + c16 of the classes kslot_row(g, j)).  Classes
// past C are zero rows with a bias of -inf, so the passes over them test no
// bounds.
__global__ __launch_bounds__(256) void pack_operands(Weights w, int count, uint4* frags, const float* O,
                                                     const float* cb, int C, int c_tiles, uint4* oa, uint4* ot,
                                                     float* cbp) {
  const int f = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, c16 = lane & 15, g = lane >> 4;
  bf16x8 v;
  if (f < count) {
    const float* W;
    int cols, ks_n, at;
    bool tr = false;
    if (f < kFrag2) {
      W = w.W1, cols = kHid, ks_n = kInPad / 32, at = f - kFrag1;
    } else if (f < kFrag3) {
      W = w.W2, cols = kHid, ks_n = kHid / 32, at = f - kFrag2;
    } else if (f < kFragT3) {
      W = w.W3, cols = kEmb, ks_n = kHid / 32, at = f - kFrag3;
    } else if (f < kFragT2) {
      W = w.W3, cols = kEmb, ks_n = kEmb / 32, at = f - kFragT3, tr = true;
    } else if (f < kFragT1) {
      W = w.W2, cols = kHid, ks_n = kHid / 32, at = f - kFragT2, tr = true;
    } else {
      W = w.W1, cols = kHid, ks_n = kHid / 32, at = f - kFragT1, tr = true;
    }
    const int col = (at / ks_n) * 16 + c16, k0 = (at % ks_n) * 32 + g * 8;
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = (__bf16)(tr ? W[(size_t)col * cols + k0 + t] : W[(size_t)(k0 + t) * cols + col]);
    frags[(size_t)f * 64 + lane] = __builtin_bit_cast(uint4, v);
  } else if (f - count < c_tiles) {
    const int ct = f - count, cls = ct * 16 + c16;
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = (__bf16)(cls < C ? O[(size_t)cls * kEmb + 8 * g + t] : 0.f);
    oa[(size_t)ct * 64 + lane] = __builtin_bit_cast(uint4, v);
    if (lane < 16) cbp[cls] = cls < C ? cb[cls] : -INFINITY;
  } else if (f - count < 2 * c_tiles) {
    const int q = f - count - c_tiles, c0 = (q >> 1) * 32, e = q & 1;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int cls = c0 + kslot_row(g, j);
      v[j] = (__bf16)(cls < C ? O[(size_t)cls * kEmb + 16 * e + c16] : 0.f);
    }
    ot[(size_t)q * 64 + lane] = __builtin_bit_cast(uint4, v);
  }
}

// One layer of 16 rows held in LDS as BF16 (`stride` values a row): the 16x16
// tile of columns 16 ct.. of the product.  `chunked` sums 64-deep partial
// products instead of one chain over K.
template <int KS>
__device__ __forceinline__ f32x4 layer_tile(const __bf16* rows, int stride, const uint4* __restrict__ frags, int ct,
                                            int lane, bool chunked) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f}, sum = {0.f, 0.f, 0.f, 0.f};
  uint4 b[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) b[ks] = frags[(size_t)(ct * KS + ks) * 64 + lane];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(rows + (lane & 15) * stride + ks * 32 + (lane >> 4) * 8);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, b[ks]), acc, 0, 0, 0);
    if (chunked && (ks & 1)) {
      for (int i = 0; i < 4; ++i) sum[i] += acc[i];
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  return chunked ? sum : acc;
}

// 16 samples per workgroup, each wave two of a layer's eight column tiles; the
// activations pass from layer to layer through LDS in the BF16 the next product
// takes.  A layer is a few MFMAs behind one round of weight loads from L2, so
// the kernel is latency-bound and small workgroups spread it over the chip:
// 1,024 samples took 75 us in seven launches (gather, three products with
// zeroing, three bias passes) and take 12.  TRAIN also stores what the backward
// pass reads (FP32).  Rows from chunk_from on accumulate the first two layers in
// 64-deep partial products, and the third always does: the order of the K-split
// products of batches that small, kept so that results stay what they were.
constexpr int kRowTile = 16;
constexpr int kXStride = kInPad + 8, kHStride = kHid + 8, kQStride = kEmb + 8;  // LDS rows start in different banks

template <bool TRAIN>
__global__ __launch_bounds__(256) void trunk_forward(const rtx_mlp_sample* __restrict__ samples, int n,
                                                     const float* __restrict__ E, int none, Weights w,
                                                     const uint4* __restrict__ frags, int chunk_from, float* X,
                                                     float* H1, float* H2, float* Q, uint4* qa, uint4* qt) {
  __shared__ __attribute__((aligned(16))) __bf16 xs[kRowTile * kXStride], h1s[kRowTile * kHStride],
      h2s[kRowTile * kHStride], qs[TRAIN ? kRowTile * kQStride : 8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, g = lane >> 4;
  const int r0 = blockIdx.x * kRowTile;
  const bool chunked = r0 >= chunk_from;
  {
    // 16 threads per sample, 12 columns each
    const int row = threadIdx.x >> 4, c0 = (threadIdx.x & 15) * 12;
    const int i = r0 + row;
    rtx_mlp_sample sm{};
    if (i < n) sm = samples[i];
    // out-of-range treelets read the "none" row
    if (sm.cur > (uint32_t)none) sm.cur = none;
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      const int c = c0 + k;
      float v = 0.f;
      if (c < 32) {
        v = E[(size_t)sm.cur * kEmb + c];
      } else if (c < 40) {
        v = (uint32_t)(c - 32) == sm.octant ? 1.f : 0.f;
      } else if (c == 40) {
        v = sm.depth;
      } else if (c < kIn) {
        const int h = (c - 41) / 32, e = (c - 41) % 32;
        const uint32_t t = h == 0 ? sm.hist[0] : h == 1 ? sm.hist[1] : h == 2 ? sm.hist[2] : sm.hist[3];
        v = E[(size_t)(t > (uint32_t)none ? (uint32_t)none : t) * kEmb + e];
      }
      if (i >= n) v = 0.f;
      xs[row * kXStride + c] = (__bf16)v;
      if (TRAIN && i < n) X[(size_t)i * kInPad + c] = v;
    }
  }
  __syncthreads();
  for (int q = 0; q < 2; ++q) {
    const int col = (2 * wave + q) * 16 + c16;
    const f32x4 z = layer_tile<kInPad / 32>(xs, kXStride, frags + kFrag1 * 64, 2 * wave + q, lane, chunked);
    const float bias = w.b1[col];
    for (int i = 0; i < 4; ++i) {
      const float v = z[i] + bias, h = v > 0.f ? v : 0.f;
      h1s[(4 * g + i) * kHStride + col] = (__bf16)h;
      if (TRAIN && r0 + 4 * g + i < n) H1[(size_t)(r0 + 4 * g + i) * kHid + col] = h;
    }
  }
  __syncthreads();
  for (int q = 0; q < 2; ++q) {
    const int col = (2 * wave + q) * 16 + c16;
    const f32x4 z = layer_tile<kHid / 32>(h1s, kHStride, frags + kFrag2 * 64, 2 * wave + q, lane, chunked);
    const float bias = w.b2[col];
    for (int i = 0; i < 4; ++i) {
      const float v = z[i] + bias, h = v > 0.f ? v : 0.f;
      h2s[(4 * g + i) * kHStride + col] = (__bf16)h;
      if (TRAIN && r0 + 4 * g + i < n) H2[(size_t)(r0 + 4 * g + i) * kHid + col] = h;
    }
  }
  __syncthreads();
  if (wave < kEmb / 16) {
    const int col = wave * 16 + c16;
    const f32x4 z = layer_tile<kHid / 32>(h2s, kHStride, frags + kFrag3 * 64, wave, lane, true);
    const float bias = w.b3[col];
    for (int i = 0; i < 4; ++i) {
      const bool in = r0 + 4 * g + i < n;
      const float q = z[i] + bias;
      if (in) Q[(size_t)(r0 + 4 * g + i) * kEmb + col] = q;
      if (TRAIN) qs[(4 * g + i) * kQStride + col] = (__bf16)(in ? q : 0.f);
    }
  }
  if constexpr (TRAIN) {
    // the queries as the output layer's operands, both orientations (see
    // pack_operands; rows past n are zero)
    __syncthreads();
    if (wave == 0) {
      qa[(size_t)blockIdx.x * 64 + lane] = *reinterpret_cast<const uint4*>(qs + c16 * kQStride + 8 * g);
    } else if (wave < 3) {
      const int e = wave - 1;
      __bf16 v[4];
      for (int j = 0; j < 4; ++j) v[j] = qs[(4 * g + j) * kQStride + 16 * e + c16];
      uint2* dst = reinterpret_cast<uint2*>(qt + (size_t)((blockIdx.x >> 1) * 2 + e) * 64 + lane) + (blockIdx.x & 1);
      *dst = *reinterpret_cast<uint2*>(v);
    }
  }
}

// ---- elementwise and reductions ---------------------------------------------------
// One Adam update.  Embedding rows never named by a sample have zero gradients
// and moments, so their update is exactly zero and only their flag is read:
// eight lanes per row, then the other parameters.  `clear` leaves the gradients
// zero for the next batch.  Bound by HBM and the last-level cache: seven or
// eight 4-byte streams over what has been touched.  7.0M parameters (200,000
// treelets, a fifth of them named within an epoch of 65,700 samples): 28 us after
// an 8 us clear -> 16 us.
__device__ __forceinline__ void adam_one(float& p, float g, float& m, float& v, float lr, float b1, float b2, float eps,
                                         float c1, float c2) {
  m = b1 * m + (1.f - b1) * g;
  v = b2 * v + (1.f - b2) * g * g;
  p -= lr * (m / c1) / (sqrtf(v / c2) + eps);
}

__global__ __launch_bounds__(256) void adam_step(float* p, float* g, float* m, float* v, const uint8_t* touched,
                                                 size_t rows, size_t count, int clear, float lr, float b1, float b2,
                                                 float eps, float c1, float c2) {
  const size_t quads = (count + 3) / 4, row_quads = rows * (kEmb / 4);
  for (size_t q = blockIdx.x * (size_t)256 + threadIdx.x; q < quads; q += (size_t)gridDim.x * 256) {
    if (q < row_quads && !touched[q / (kEmb / 4)]) continue;
    if (q * 4 + 4 <= count) {
      float4 P = reinterpret_cast<float4*>(p)[q], M = reinterpret_cast<float4*>(m)[q], V = reinterpret_cast<float4*>(v)[q];
      const float4 G = reinterpret_cast<float4*>(g)[q];
      adam_one(P.x, G.x, M.x, V.x, lr, b1, b2, eps, c1, c2);
      adam_one(P.y, G.y, M.y, V.y, lr, b1, b2, eps, c1, c2);
      adam_one(P.z, G.z, M.z, V.z, lr, b1, b2, eps, c1, c2);
      adam_one(P.w, G.w, M.w, V.w, lr, b1, b2, eps, c1, c2);
      reinterpret_cast<float4*>(p)[q] = P;
      reinterpret_cast<float4*>(m)[q] = M;
      reinterpret_cast<float4*>(v)[q] = V;
      if (clear) reinterpret_cast<float4*>(g)[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
      for (size_t k = q * 4; k < count; ++k) {
        adam_one(p[k], g[k], m[k], v[k], lr, b1, b2, eps, c1, c2);
        if (clear) g[k] = 0.f;
      }
    }
  }
}

// ---- trunk backward ---------------------------------------------------------------
// dq -> dh2 -> dh1 -> dx for 16 samples per workgroup, as trunk_forward goes
// forward: dh2 and dh1 are stored for the weight gradients, the bias gradients
// are column sums, and dx goes straight into the embedding rows it came from.
// Samples of a workgroup that name the same row add up in LDS first: the
// ancestors in the history are shared by most samples, and one atomic per
// sample on those rows would serialise.  1,024 samples: 96 us in eleven launches
// (products with zeroing, masks, column sums, a scatter over 160 passes) -> 12.
struct Gradients {
  float *E, *b1, *b2, *b3;
};

__global__ __launch_bounds__(256) void trunk_backward(const rtx_mlp_sample* __restrict__ samples, int n, int none,
                                                      const uint4* __restrict__ frags, const float* __restrict__ dQ,
                                                      const float* __restrict__ H1, const float* __restrict__ H2,
                                                      float* dH1, float* dH2, Gradients G, uint8_t* touched) {
  __shared__ __attribute__((aligned(16))) __bf16 qs[kRowTile * kQStride], h2s[kRowTile * kHStride],
      h1s[kRowTile * kHStride];
  __shared__ float xs[kRowTile * (kInPad + 4)];
  __shared__ uint32_t rows[5][kRowTile], same[5][kRowTile];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, g = lane >> 4;
  const int r0 = blockIdx.x * kRowTile;
  if (threadIdx.x < 5 * kRowTile) {
    const int h = threadIdx.x / kRowTile, i = threadIdx.x % kRowTile;
    uint32_t t = 0xffffffffu;
    if (r0 + i < n) {
      const rtx_mlp_sample& sm = samples[r0 + i];
      t = h == 0 ? sm.cur : sm.hist[h - 1];
      if (t > (uint32_t)none) t = (uint32_t)none;  // as the forward pass reads it
    }
    rows[h][i] = t;
  }
  {
    // two rows per wave and pass
    float sum = 0.f;
    const int col = threadIdx.x % kEmb;
    for (int row = threadIdx.x / kEmb; row < kRowTile; row += 8) {
      const float v = r0 + row < n ? dQ[(size_t)(r0 + row) * kEmb + col] : 0.f;
      qs[row * kQStride + col] = (__bf16)v;
      sum += v;
    }
    xs[threadIdx.x] = sum;
  }
  __syncthreads();
  if (threadIdx.x < kEmb) {
    float sum = 0.f;
    for (int k = 0; k < 8; ++k) sum += xs[k * kEmb + threadIdx.x];
    atomicAdd(&G.b3[threadIdx.x], sum);
  } else if (threadIdx.x >= 64 && threadIdx.x < 64 + 5 * kRowTile) {
    // the samples that name this one's row, none when an earlier one does
    const int h = (threadIdx.x - 64) / kRowTile, i = (threadIdx.x - 64) % kRowTile;
    const uint32_t t = rows[h][i];
    uint32_t m = 0;
    for (int k = 0; k < kRowTile; ++k) m |= rows[h][k] == t ? 1u << k : 0u;
    same[h][i] = t == 0xffffffffu || (m & ((1u << i) - 1u)) ? 0u : m;
  }
  // masks a layer's tile where its activation was clipped, stores it, adds its column sums
  auto finish = [&](f32x4 z, int col, const float* H, float* dH, __bf16* lds, float* gb) {
    float sum = 0.f;
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + 4 * g + i;
      float v = 0.f;
      if (r < n) {
        v = H[(size_t)r * kHid + col] > 0.f ? z[i] : 0.f;
        dH[(size_t)r * kHid + col] = v;
      }
      lds[(4 * g + i) * kHStride + col] = (__bf16)v;
      sum += v;
    }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (g == 0) atomicAdd(&gb[col], sum);
  };
  for (int q = 0; q < 2; ++q) {
    const int ct = 2 * wave + q;
    finish(layer_tile<kEmb / 32>(qs, kQStride, frags + kFragT3 * 64, ct, lane, false), ct * 16 + c16, H2, dH2, h2s, G.b2);
  }
  __syncthreads();
  for (int q = 0; q < 2; ++q) {
    const int ct = 2 * wave + q;
    finish(layer_tile<kHid / 32>(h2s, kHStride, frags + kFragT2 * 64, ct, lane, false), ct * 16 + c16, H1, dH1, h1s, G.b1);
  }
  __syncthreads();
  for (int q = 0; q < 3; ++q) {
    const int ct = 3 * wave + q;
    const f32x4 z = layer_tile<kHid / 32>(h1s, kHStride, frags + kFragT1 * 64, ct, lane, false);
    for (int i = 0; i < 4; ++i) xs[(4 * g + i) * (kInPad + 4) + ct * 16 + c16] = z[i];
  }
  __syncthreads();
  // 32 threads per (slot, sample): the first sample that names a row adds it for all
  const int e = threadIdx.x & 31;
  for (int it = threadIdx.x >> 5; it < 5 * kRowTile; it += 8) {
    const int h = it / kRowTile, i = it % kRowTile;
    uint32_t m = same[h][i];
    if (m == 0) continue;
    const uint32_t t = rows[h][i];
    const int col = h == 0 ? e : 41 + (h - 1) * kEmb + e;
    float sum = 0.f;
    for (; m; m &= m - 1) sum += xs[(__ffs((int)m) - 1) * (kInPad + 4) + col];
    atomicAdd(&G.E[(size_t)t * kEmb + e], sum);
    if (e == 0) touched[t] = 1;
  }
}

// The three weight gradients A^T B over the batch's rows in one launch: 32 x 32
// output tiles (24 of W1, 16 of W2, 4 of W3) by row ranges.  A workgroup's four
// waves take every fourth 32-row step and add up in LDS, so an output element
// takes one atomic per row range.  1,024 rows: 28 us in three launches -> 9; at
// ranges of 256 rows, with two serial steps per wave, 16.
struct WeightGrad {
  const float *A, *B;
  float* C;
  int lda, ldb;
};

__global__ __launch_bounds__(256) void weight_grads(WeightGrad w1, WeightGrad w2, WeightGrad w3, int n, int rows_per) {
  __shared__ float red[3][64 * 17];
  const int id = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, g = lane >> 4;
  const WeightGrad w = id < 24 ? w1 : id < 40 ? w2 : w3;
  const int tile = id < 24 ? id : id < 40 ? id - 24 : (id - 40) * 4;
  const int m0 = (tile / 4) * 32, n0 = (tile % 4) * 32;
  const int rend = min(n, (int)(blockIdx.y + 1) * rows_per);
  f32x4 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = blockIdx.y * rows_per + wave * 32; k0 < rend; k0 += 128) {
    bf16x8 a[2], b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int k = k0 + g * 8 + t;
        a[i][t] = (__bf16)(k < rend ? w.A[(size_t)k * w.lda + m0 + i * 16 + c16] : 0.f);
        b[i][t] = (__bf16)(k < rend ? w.B[(size_t)k * w.ldb + n0 + i * 16 + c16] : 0.f);
      }
    for (int i = 0; i < 2; ++i)
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
  }
  if (wave > 0)
    for (int q = 0; q < 16; ++q) red[wave - 1][lane * 17 + q] = acc[q >> 3][(q >> 2) & 1][q & 3];
  __syncthreads();
  if (wave == 0)
    for (int q = 0; q < 16; ++q) {
      const float v = ((acc[q >> 3][(q >> 2) & 1][q & 3] + red[0][lane * 17 + q]) + red[1][lane * 17 + q]) + red[2][lane * 17 + q];
      atomicAdd(&w.C[(size_t)(m0 + (q >> 3) * 16 + 4 * g + (q & 3)) * w.ldb + n0 + ((q >> 2) & 1) * 16 + c16], v);
    }
}

// ---- fused output layer ----------------------------------------------------------
// The logits L = Q O^T + o (Q: [n x 32] queries, O: [C x 32] class vectors, o the
// class biases) exist only as 16x16 MFMA tiles in registers.  ce_stats keeps each
// row's running maximum and exp-sum over a chunk of classes; ce_finish turns the
// chunks into the row's log-sum-exp and the loss; ce_grad recomputes the tiles to
// form dL = (softmax - onehot) / n, once per 32 classes for dO = dL^T Q and the
// bias gradient, once per 32 rows for dQ = dL O.  The sum over k inside one MFMA
// does not depend on which k-slot holds which term, so a dL tile left in the
// result layout (lane = column, rows 4g..4g+3 of lane group g = lane / 16) feeds
// the next MFMA as it is: k-slot 8g + j pairs tile row 4g + j (j < 4) of the
// first 16-row tile with the same k-slot of the other operand, and 4g + j - 4 of
// the second tile for j >= 4.
//
// Every operand comes from a packed fragment (pack_operands, trunk_forward), one
// 16-byte load per lane from L2, used for two tiles: rows staged through LDS had
// cost sixteen 2-byte LDS reads per lane and 32 classes for the transposed
// operand, the FP32 conversions again in each workgroup and two barriers per
// stage.  1,024 rows x 16,384 classes: statistics 28 -> 16 us, both gradients 54
// -> 31 us.  Bound by VALU work on each logit, the exponential above all.
constexpr int kCeChunk = 256;  // classes per ce_stats wave
constexpr int kCeCls = 128;    // classes per LDS stage of logits_top4
constexpr int kCeRange = 512;  // classes per ce_grad wave that sums dQ

// Eight FP32 values rounded to BF16 (round to nearest even, as the MFMA operand
// loads of gemm_bf16), packed into 16 bytes.
__device__ __forceinline__ uint4 pack_bf16x8(const float* __restrict__ p) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 b = *reinterpret_cast<const float4*>(p + 4);
  bf16x8 v;
  v[0] = (__bf16)a.x; v[1] = (__bf16)a.y; v[2] = (__bf16)a.z; v[3] = (__bf16)a.w;
  v[4] = (__bf16)b.x; v[5] = (__bf16)b.y; v[6] = (__bf16)b.z; v[7] = (__bf16)b.w;
  return __builtin_bit_cast(uint4, v);
}

// Row r of an [rows x 32] FP32 matrix, elements k0..k0+7, as BF16 (zero past `rows`).
__device__ __forceinline__ bf16x8 ld_row8(const float* __restrict__ M, int rows, int r, int k0) {
  if (r < rows) return __builtin_bit_cast(bf16x8, pack_bf16x8(M + (size_t)r * kEmb + k0));
  return __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
}

// Rows [r0, r0 + count) of an [rows x 32] FP32 matrix into LDS as BF16: row i
// at S[4 * i .. 4 * i + 3] (16 bytes = 8 values each).  Every thread of the block calls it.
__device__ __forceinline__ void stage_rows(uint4* S, const float* __restrict__ M, int r0, int count) {
  for (int u = threadIdx.x; u < count * 4; u += blockDim.x) S[u] = pack_bf16x8(M + (size_t)(r0 + u / 4) * kEmb + (u % 4) * 8);
}

__device__ __forceinline__ bf16x8 lds_row8(const uint4* S, int i, int g, bool valid) {
  return __builtin_bit_cast(bf16x8, valid ? S[4 * i + g] : make_uint4(0, 0, 0, 0));
}

__device__ __forceinline__ bf16x8 frag(const uint4* __restrict__ f, int at, int lane) {
  return __builtin_bit_cast(bf16x8, f[(size_t)at * 64 + lane]);
}

// e^d for the terms of the prediction's softmax: for h near d log2(e), e^d is
// 2^h (1 + r) but for r^2, where r = d - h ln(2) comes exactly from two FMAs (ln(2) in
// two parts).  h is taken 8e-6 below the product, more than its rounding, so r lies in
// [0, 2e-5] and the FMA's clamp to [0, 1], which costs nothing, only touches terms
// below 1e-37 and those where h overflows (d of -inf among them): r is no number there,
// and the clamp makes it 0.  For d in [-80, 32] the relative error is at most 1.4e-7,
// 3.7e-8 in the mean square (expf 8.4e-8 and 2.7e-8); one product and 2^x alone had
// 1e-7 |d|, with d up to 32 (see logits_top4).  Probabilities against 64 bits are as with
// expf (1e-7; a class 20 or 28 above the rest 8e-7, with the product alone 1.2e-6).
// 20,011 rows of 16,384 classes take 253 us with the product alone and 268 so; with expf,
// whose range handling takes a dozen more instructions, 326 beside 257.  Training takes
// expf: there each term is a gradient of its own.
__device__ __forceinline__ float exp_term(float d) {
  const float h = __builtin_fmaf(d, 1.44269504088896340736f, -8e-6f);
  float r = __builtin_fmaf(h, -0x1.62e430p-1f, d);
  r = __builtin_fmaf(h, 0x1.05c610p-29f, r);
  const float e = __builtin_amdgcn_exp2f(h);
  return __builtin_fmaf(e, __builtin_amdgcn_fmed3f(r, 0.f, 1.f), e);
}

// (m, s) <- the log-sum-exp pair of the union of two sets: max and exp-sum relative to it.
// The maximum of no logits is kLowest, which no finite one is below: terms of -inf (and
// of padding) are 0 relative to it, and a NaN makes the sum NaN wherever it stands.
constexpr float kLowest = -FLT_MAX;
__device__ __forceinline__ void lse_merge(float& m, float& s, float m2, float s2) {
  const float mx = fmaxf(m, m2);
  s = s * expf(m - mx) + s2 * expf(m2 - mx);
  m = mx;
}

// One wave: 32 rows x kCeChunk classes, the classes as the MFMA's rows, so a lane
// holds four logits of one sample per tile.  pm/ps[r * nchunk + chunk] get the
// row's maximum logit and its exp-sum over the chunk.  grid.x: 32-row groups,
// grid.y: four chunks per workgroup.
__global__ __launch_bounds__(256) void ce_stats(const uint4* __restrict__ qa, int n, const uint4* __restrict__ oa,
                                                const float* __restrict__ cbp, int c_tiles, int nchunk, float* pm,
                                                float* ps) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int chunk = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (chunk >= nchunk) return;
  const bf16x8 b[2] = {frag(qa, 2 * blockIdx.x, lane), frag(qa, 2 * blockIdx.x + 1, lane)};
  float m[2] = {kLowest, kLowest}, s[2] = {0.f, 0.f};
  const int t0 = chunk * (kCeChunk / 16), t1 = min(c_tiles, t0 + kCeChunk / 16);
  for (int ct = t0; ct < t1; ++ct) {
    const bf16x8 a = frag(oa, ct, lane);
    const float4 bias = *reinterpret_cast<const float4*>(cbp + ct * 16 + 4 * g);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[k], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      const float x0 = acc[0] + bias.x, x1 = acc[1] + bias.y, x2 = acc[2] + bias.z, x3 = acc[3] + bias.w;
      const float mx = fmaxf(fmaxf(x0, x1), fmaxf(x2, x3));
      if (mx > m[k]) {
        s[k] *= expf(m[k] - mx);
        m[k] = mx;
      }
      s[k] += (expf(x0 - m[k]) + expf(x1 - m[k])) + (expf(x2 - m[k]) + expf(x3 - m[k]));
    }
  }
  // the four lane groups hold quarters of the chunk's classes
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    for (int o = 16; o < 64; o <<= 1) {
      const float m2 = __shfl_xor(m[k], o, 64), s2 = __shfl_xor(s[k], o, 64);
      lse_merge(m[k], s[k], m2, s2);
    }
    const int r = (2 * blockIdx.x + k) * 16 + c16;
    if (g == 0 && r < n) {
      pm[(size_t)r * nchunk + chunk] = m[k];
      ps[(size_t)r * nchunk + chunk] = s[k];
    }
  }
}

// One wave per row: log-sum-exp over the chunks, the target and its logit (the
// BF16-rounded product in FP32), the loss, and dQ cleared.  Rows past n, up to
// a multiple of 32, get an infinite log-sum-exp: their dL is zero.
__global__ __launch_bounds__(256) void ce_finish(const float* pm, const float* ps, int nchunk,
                                                 const float* __restrict__ Q, const float* __restrict__ O,
                                                 const float* __restrict__ cb, const rtx_mlp_sample* samples, int n,
                                                 int C, float inv_n, float* lse, uint32_t* target, float* loss,
                                                 float* dQ) {
  __shared__ float part[4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = blockIdx.x * 4 + w;
  float nll = 0.f;
  if (r < n) {
    float m = kLowest, sm = 0.f;
    for (int c = lane; c < nchunk; c += 64) lse_merge(m, sm, pm[(size_t)r * nchunk + c], ps[(size_t)r * nchunk + c]);
    for (int o = 32; o > 0; o >>= 1) {
      const float m2 = __shfl_xor(m, o, 64), s2 = __shfl_xor(sm, o, 64);
      lse_merge(m, sm, m2, s2);
    }
    const uint32_t t = samples[r].target;
    float x = 0.f;
    if (lane < kEmb) {
      if (t < (uint32_t)C) x = (float)(__bf16)Q[(size_t)r * kEmb + lane] * (float)(__bf16)O[(size_t)t * kEmb + lane];
      dQ[(size_t)r * kEmb + lane] = 0.f;
    }
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    const float l = m + logf(sm);
    if (t < (uint32_t)C) nll = (l - (x + cb[t])) * inv_n;
    if (lane == 0) {
      lse[r] = l;
      target[r] = t;
    }
  } else if (lane == 0) {
    lse[r] = INFINITY;
    target[r] = 0xffffffffu;
  }
  if (lane == 0) part[w] = nll;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(loss, (part[0] + part[1]) + (part[2] + part[3]));
}

// dL of one logit: (softmax - onehot) / n.
__device__ __forceinline__ float ce_dl(float logit, float bias, float lse, bool hot, float inv_n) {
  return (expf(logit + bias - lse) - (hot ? 1.f : 0.f)) * inv_n;
}

// Two kinds of workgroup in one launch, so that both fill the chip together.
// The first ceil(C / 32) sum 32 classes' dO and bias gradient: their four waves
// take every fourth 32-row step and add up in LDS, so each class is written once.
// The others sum 32 rows' dQ over four ranges of kCeRange classes, one per wave,
// added up in LDS and then atomically (dQ cleared by ce_finish).
struct CeGrad {
  const uint4 *qa, *qt, *oa, *ot;
  const float *cbp, *lse;
  const uint32_t* target;
  int n, row_steps, C, c_steps, q_blocks;  // q_blocks: workgroups per 32 rows
  float inv_n;
  float *gO, *gc, *dQ;
};

__global__ __launch_bounds__(256) void ce_grad(CeGrad p) {
  __shared__ float red[3][64 * 17];
  __shared__ float redc[3][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c16 = lane & 15;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 d[2][2] = {{zero, zero}, {zero, zero}};  // [tile of 16 classes / rows][half of the embedding]
  const bool by_class = blockIdx.x < (uint32_t)p.c_steps;
  const int at = by_class ? blockIdx.x : (blockIdx.x - p.c_steps) / p.q_blocks;  // 32 classes / 32 rows
  float dc[2] = {0.f, 0.f};
  if (by_class) {
    const bf16x8 b[2] = {frag(p.oa, 2 * at, lane), frag(p.oa, 2 * at + 1, lane)};
    const float bias[2] = {p.cbp[at * 32 + c16], p.cbp[at * 32 + 16 + c16]};
    const uint32_t cls[2] = {(uint32_t)(at * 32 + c16), (uint32_t)(at * 32 + 16 + c16)};
    for (int st = wave; st < p.row_steps; st += 4) {
      const bf16x8 a[2] = {frag(p.qa, 2 * st, lane), frag(p.qa, 2 * st + 1, lane)};
      const bf16x8 t0 = frag(p.qt, 2 * st, lane), t1 = frag(p.qt, 2 * st + 1, lane);
      float4 l[2];
      uint4 t[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        l[h] = *reinterpret_cast<const float4*>(p.lse + st * 32 + h * 16 + 4 * g);
        t[h] = *reinterpret_cast<const uint4*>(p.target + st * 32 + h * 16 + 4 * g);
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        bf16x8 v;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h], b[k], zero, 0, 0, 0);
          const float x[4] = {ce_dl(acc[0], bias[k], l[h].x, t[h].x == cls[k], p.inv_n),
                              ce_dl(acc[1], bias[k], l[h].y, t[h].y == cls[k], p.inv_n),
                              ce_dl(acc[2], bias[k], l[h].z, t[h].z == cls[k], p.inv_n),
                              ce_dl(acc[3], bias[k], l[h].w, t[h].w == cls[k], p.inv_n)};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            dc[k] += x[i];
            v[4 * h + i] = (__bf16)x[i];
          }
        }
        // dO tile [16 classes x 16 emb] += dL^T (classes x 32 rows) . Q (32 rows x 16 emb)
        d[k][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, t0, d[k][0], 0, 0, 0);
        d[k][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, t1, d[k][1], 0, 0, 0);
      }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      dc[k] += __shfl_xor(dc[k], 16, 64);
      dc[k] += __shfl_xor(dc[k], 32, 64);
    }
    if (wave > 0 && g < 2) redc[wave - 1][g * 16 + c16] = g ? dc[1] : dc[0];
  } else {
    const bf16x8 b[2] = {frag(p.qa, 2 * at, lane), frag(p.qa, 2 * at + 1, lane)};  // columns of the transposed logits
    const float l[2] = {p.lse[at * 32 + c16], p.lse[at * 32 + 16 + c16]};
    const uint32_t t[2] = {p.target[at * 32 + c16], p.target[at * 32 + 16 + c16]};
    const int s0 = (((blockIdx.x - p.c_steps) % p.q_blocks) * 4 + wave) * (kCeRange / 32);
    const int s1 = min(p.c_steps, s0 + kCeRange / 32);
    for (int st = s0; st < s1; ++st) {
      const bf16x8 a[2] = {frag(p.oa, 2 * st, lane), frag(p.oa, 2 * st + 1, lane)};
      const bf16x8 t0 = frag(p.ot, 2 * st, lane), t1 = frag(p.ot, 2 * st + 1, lane);
      float4 bias[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) bias[h] = *reinterpret_cast<const float4*>(p.cbp + st * 32 + h * 16 + 4 * g);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        bf16x8 v;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h], b[k], zero, 0, 0, 0);
          const uint32_t c0 = (uint32_t)(st * 32 + h * 16 + 4 * g);
          v[4 * h] = (__bf16)ce_dl(acc[0], bias[h].x, l[k], t[k] == c0, p.inv_n);
          v[4 * h + 1] = (__bf16)ce_dl(acc[1], bias[h].y, l[k], t[k] == c0 + 1, p.inv_n);
          v[4 * h + 2] = (__bf16)ce_dl(acc[2], bias[h].z, l[k], t[k] == c0 + 2, p.inv_n);
          v[4 * h + 3] = (__bf16)ce_dl(acc[3], bias[h].w, l[k], t[k] == c0 + 3, p.inv_n);
        }
        // dQ^T tile [16 emb x 16 rows] += O^T (emb x 32 classes) . dL^T (32 classes x rows)
        d[k][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t0, v, d[k][0], 0, 0, 0);
        d[k][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t1, v, d[k][1], 0, 0, 0);
      }
    }
  }
  if (wave > 0)
    for (int q = 0; q < 16; ++q) red[wave - 1][lane * 17 + q] = d[q >> 3][(q >> 2) & 1][q & 3];
  __syncthreads();
  if (wave > 0) return;
  for (int q = 0; q < 16; ++q) {
    const int k = q >> 3, e = (q >> 2) & 1, i = q & 3;
    const float v = ((d[k][e][i] + red[0][lane * 17 + q]) + red[1][lane * 17 + q]) + red[2][lane * 17 + q];
    if (by_class) {
      // result layout: emb column c16 (+16), classes 4g + i
      const int c = at * 32 + k * 16 + 4 * g + i;
      if (c < p.C) p.gO[(size_t)c * kEmb + e * 16 + c16] = v;
    } else {
      // result layout: row column c16, emb 4g + i (+16)
      const int r = at * 32 + k * 16 + c16;
      if (r < p.n) atomicAdd(&p.dQ[(size_t)r * kEmb + e * 16 + 4 * g + i], v);
    }
  }
  if (by_class && g < 2) {
    const int c = at * 32 + g * 16 + c16;
    const float v = ((g ? dc[1] : dc[0]) + redc[0][g * 16 + c16]) + (redc[1][g * 16 + c16] + redc[2][g * 16 + c16]);
    if (c < p.C) p.gc[c] = v;
  }
}

// ---- prediction: top-4 classes and probabilities ------------------------------------
// The best four of a set of logits, best first, ties to the lower class (-1:
// none), with the set's maximum and exp-sum relative to it.
struct Top4 {
  float v[4];
  int c[4];
  float m, s;
};
static_assert(sizeof(Top4) == 40, "partial results are stored as Top4");

// x into the list, when it is greater than the last one; classes come in ascending
// order, so an equal value stays behind.  No branches: 15 instructions.
__device__ __forceinline__ void top4_insert(Top4& t, float x, int c) {
  const bool b0 = x > t.v[0], b1 = x > t.v[1], b2 = x > t.v[2], b3 = x > t.v[3];
  auto pick = [](bool b, int a, int other) { return b ? a : other; };
  t.c[3] = pick(b2, t.c[2], pick(b3, c, t.c[3]));
  t.c[2] = pick(b1, t.c[1], pick(b2, c, t.c[2]));
  t.c[1] = pick(b0, t.c[0], pick(b1, c, t.c[1]));
  t.c[0] = pick(b0, c, t.c[0]);
  t.v[3] = __builtin_amdgcn_fmed3f(t.v[2], t.v[3], x);
  t.v[2] = __builtin_amdgcn_fmed3f(t.v[1], t.v[2], x);
  t.v[1] = __builtin_amdgcn_fmed3f(t.v[0], t.v[1], x);
  t.v[0] = b0 ? x : t.v[0];
}

__device__ __forceinline__ bool top4_before(float v, int c, float v2, int c2) {
  return c >= 0 && (c2 < 0 || v > v2 || (v == v2 && c < c2));
}

// t <- the four best of both, and (top4_merge) the exp-sum of the union
__device__ __forceinline__ void top4_merge_lists(Top4& t, const Top4& o) {
  // Both are sorted, so the four best of the union are the better of t[k] and
  // o[3 - k] for each k; two exchange steps order them.
  float v[4];
  int c[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const bool keep = top4_before(t.v[k], t.c[k], o.v[3 - k], o.c[3 - k]);
    v[k] = keep ? t.v[k] : o.v[3 - k];
    c[k] = keep ? t.c[k] : o.c[3 - k];
  }
  auto order = [&](int a, int b) {
    if (top4_before(v[b], c[b], v[a], c[a])) {
      const float tv = v[a];
      const int tc = c[a];
      v[a] = v[b];
      c[a] = c[b];
      v[b] = tv;
      c[b] = tc;
    }
  };
  order(0, 2);
  order(1, 3);
  order(0, 1);
  order(2, 3);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    t.v[k] = v[k];
    t.c[k] = c[k];
  }
}

__device__ __forceinline__ void top4_merge(Top4& t, const Top4& o) {
  top4_merge_lists(t, o);
  lse_merge(t.m, t.s, o.m, o.s);
}

// One block: 64 rows (a wave per 16) against the classes [y * cper, y * cper +
// cper), staged in LDS kCeCls at a time.  The MFMA's rows are classes and its
// columns the wave's samples, so a lane keeps one sample's best four over a
// quarter of the classes, in registers, and the logits are never stored: 20,011
// samples x 16,384 classes wrote and read 1.3 GB of them twice (3.4 ms in five
// products and five scans) and take 0.20 ms here.  Bound by the VALU work on each
// logit: its compare and exponential, then the insertions.  Some lane of a wave
// has a better logit in nearly every step, so the lanes only put theirs aside
// (kAside of them, in LDS) and insert together once one lane's places run out;
// inserting in each step took 0.26 ms.  A lane passes over what the same sample's
// other three lanes already have four better ones of (equal ones stay: the lower
// class wins, and only a lane's own classes come in order).  Each class split
// starts with empty lists, so there are only as many as one round of workgroups
// has room for (kPredBlocks): with two rounds, and stages of 256 classes, 0.23 ms.
// (The two alternatives were measured before exp_term was corrected, when this took
// 0.18 ms.)
constexpr int kAside = 11;
__global__ __launch_bounds__(256) void logits_top4(const float* __restrict__ Q, int n, const float* __restrict__ O,
                                                   const float* __restrict__ cb, int C, int cper, Top4* part) {
  __shared__ uint4 Os[kCeCls * 4];
  __shared__ __attribute__((aligned(16))) float cbs[kCeCls];
  const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int row = blockIdx.x * 64 + (threadIdx.x >> 6) * 16 + c16;
  const bf16x8 b = ld_row8(Q, n, row, 8 * g);
  __shared__ float aside_v[kAside][256];
  __shared__ int aside_c[kAside][256];
  Top4 t;
  for (int k = 0; k < 4; ++k) {
    t.v[k] = -INFINITY;
    t.c[k] = -1;
  }
  t.m = kLowest;
  t.s = 0.f;
  int held = 0;  // logits put aside
  float least = -INFINITY, most = -INFINITY;  // what a logit has to exceed; the greatest so far
  // insert them, and refer the exp-sum to the greatest logit
  auto insert_held = [&]() {
    for (int k = 0; __ballot(k < held); ++k) {
      const float v = aside_v[k][threadIdx.x];
      const int c = aside_c[k][threadIdx.x];
      top4_insert(t, k < held ? v : -INFINITY, c);
    }
    held = 0;
    float other = fmaxf(__shfl_xor(t.v[3], 16, 64), __shfl_xor(t.v[3], 32, 64));
    other = fmaxf(other, __shfl_xor(t.v[3], 48, 64));
    const uint32_t u = __float_as_uint(other);  // the next float below it
    const float below = __uint_as_float((int)u > 0 ? u - 1u : (u << 1) == 0u ? 0x80000001u : u + 1u);
    least = other > -INFINITY ? fmaxf(t.v[3], below) : t.v[3];
    if (most > t.m) {
      t.s *= expf(t.m - most);
      t.m = most;
    }
  };
  const int cbeg = blockIdx.y * cper, cend = min(C, cbeg + cper);
  for (int cc = cbeg; cc < cend; cc += kCeCls) {
    const int nc = min(kCeCls, cend - cc);
    __syncthreads();  // the previous stage is read
    stage_rows(Os, O, cc, nc);
    // a class past the end has a logit of -inf
    for (int i = threadIdx.x; i < kCeCls; i += blockDim.x) cbs[i] = i < nc ? cb[cc + i] : -INFINITY;
    __syncthreads();
    for (int ct = 0; ct < nc; ct += 32) {  // two tiles at a time
      float x[8];
      f32x4 acc[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_row8(Os, ct + 16 * h + c16, g, ct + 16 * h + c16 < nc), b,
                                                         f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float4 bias = *reinterpret_cast<const float4*>(cbs + ct + 16 * h + 4 * g);
        x[4 * h] = acc[h][0] + bias.x;
        x[4 * h + 1] = acc[h][1] + bias.y;
        x[4 * h + 2] = acc[h][2] + bias.z;
        x[4 * h + 3] = acc[h][3] + bias.w;
      }
      const float mx = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
      if (mx > least) {
        most = fmaxf(most, mx);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (x[i] > least) {
            aside_v[held][threadIdx.x] = x[i];
            aside_c[held][threadIdx.x] = cc + ct + 16 * (i >> 2) + 4 * g + (i & 3);
            held++;
          }
      }
      // (the exponentials stay below 2^47 by the second)
      if (__ballot(held > kAside - 8 || mx > t.m + 32.f)) {
        most = fmaxf(most, mx);
        insert_held();
      }
      t.s += ((exp_term(x[0] - t.m) + exp_term(x[1] - t.m)) + (exp_term(x[2] - t.m) + exp_term(x[3] - t.m))) +
             ((exp_term(x[4] - t.m) + exp_term(x[5] - t.m)) + (exp_term(x[6] - t.m) + exp_term(x[7] - t.m)));
    }
  }
  insert_held();
  // the four lane groups hold quarters of the same rows' classes
  for (int o = 16; o < 64; o <<= 1) {
    Top4 u;
    for (int k = 0; k < 4; ++k) {
      u.v[k] = __shfl_xor(t.v[k], o, 64);
      u.c[k] = __shfl_xor(t.c[k], o, 64);
    }
    u.m = __shfl_xor(t.m, o, 64);
    u.s = __shfl_xor(t.s, o, 64);
    top4_merge(t, u);
  }
  if (g == 0 && row < n) part[(size_t)blockIdx.y * n + row] = t;
}

// One thread per row: its class splits merged, then classes and probabilities.  The
// splits' exp-sums, of which a few rows have one per 256 classes, are referred to the
// row's maximum once each and added in FP64: a chain of FP32 merges doubled the error of
// 64 rows' probabilities over 16,384 classes (7e-8 -> 1.4e-7 for logits within 1).
__global__ __launch_bounds__(64) void top4_finish(const Top4* part, int n, int splits, uint32_t* out, float* prob) {
  const int r = blockIdx.x * 64 + threadIdx.x;
  if (r >= n) return;
  Top4 t = part[r];
  for (int k = 1; k < splits; ++k) {
    const Top4 o = part[(size_t)k * n + r];
    top4_merge_lists(t, o);
    t.m = fmaxf(t.m, o.m);
  }
  double sum = 0.0;
  for (int k = 0; k < splits; ++k) {
    const Top4& o = part[(size_t)k * n + r];
    sum += (double)o.s * (double)expf(o.m - t.m);
  }
  t.s = (float)sum;
  for (int k = 0; k < 4; ++k) out[(size_t)r * 4 + k] = t.c[k] < 0 ? RTX_NO_TREELET : (uint32_t)t.c[k];
  if (prob)
    for (int k = 0; k < 4; ++k) prob[(size_t)r * 4 + k] = t.c[k] < 0 ? 0.f : expf(t.v[k] - t.m) / t.s;
}

template <bool TA, bool TB, int BN>
hipError_t gemm_launch(hipStream_t s, int M, int N, int K, const float* A, int lda, const float* B, int ldb, float* C,
                       int ldc, int accumulate) {
  constexpr int BM = BN == 64 ? 64 : 128;
  const int tiles = ((N + BN - 1) / BN) * ((M + BM - 1) / BM);
  // split K when the output has too few tiles to fill the chip (the weight
  // gradients: a few tiles, K = the batch), down to 64-deep chunks (32 for
  // outputs of under 8 tiles)
  int split = 1;
  if (tiles < 256 && K >= 512) split = std::max(1, std::min(K / (tiles < 8 ? 32 : 64), (512 + tiles - 1) / tiles));
  // the batch-sized activations (a few dozen tiles, K 128-192): 64-deep chunks
  else if (tiles < 64 && K >= 128) split = std::max(1, std::min(K / 64, (128 + tiles - 1) / tiles));
  int k_chunk = (K + split - 1) / split;
  k_chunk = (k_chunk + 31) / 32 * 32;
  split = (K + k_chunk - 1) / k_chunk;
  if (split > 1 && !accumulate) {
    hipLaunchKernelGGL(zero_rows, dim3(256), dim3(256), 0, s, C, M, N, ldc);
  }
  dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM, split);
  hipLaunchKernelGGL((gemm_bf16<TA, TB, BN>), grid, dim3(256), 0, s, M, N, K, k_chunk, A, lda, B, ldb, C, ldc,
                     accumulate);
  return hipGetLastError();
}

template <bool TA, bool TB>
hipError_t gemm(hipStream_t s, int M, int N, int K, const float* A, int lda, const float* B, int ldb, float* C,
                int ldc, int accumulate) {
  if (N <= 32) return gemm_launch<TA, TB, 32>(s, M, N, K, A, lda, B, ldb, C, ldc, accumulate);
  return gemm_launch<TA, TB, 64>(s, M, N, K, A, lda, B, ldb, C, ldc, accumulate);
}

}  // namespace

// ---- model object -------------------------------------------------------------
struct rtx_mlp {
  rtx_ctx* ctx = nullptr;
  hipStream_t stream = nullptr;
  int device = 0;
  uint32_t T = 0, C = 0;  // embedded treelets (row T = "none"), output classes
  // parameter blocks inside one FP32 buffer
  size_t oE, oW1, ob1, oW2, ob2, oW3, ob3, oO, oc, count;
  float *P = nullptr, *G = nullptr, *M1 = nullptr, *V1 = nullptr;
  uint32_t steps = 0;
  // activations of one batch
  uint32_t cap = 0;
  float *X = nullptr, *H1 = nullptr, *H2 = nullptr, *Q = nullptr;
  float *dQ = nullptr, *dH2 = nullptr, *dH1 = nullptr, *loss = nullptr;
  // fused output layer: per-row chunk maxima and exp-sums, log-sum-exp and
  // target (rows padded to a multiple of 32), queries as MFMA operands
  float *pm = nullptr, *ps = nullptr, *lse = nullptr, *target = nullptr, *qa = nullptr, *qt = nullptr;
  // parameters as MFMA operands, packed before each pass: the trunk's weights,
  // the class vectors in both orientations and the padded class biases
  uint4 *frags = nullptr, *oa = nullptr, *ot = nullptr;
  float* cbp = nullptr;
  // embedding rows that ever had a gradient (one byte each)
  uint8_t* touched = nullptr;
  // prediction: queries and per-split results of one chunk of rows
  float* pred_q = nullptr;
  Top4* pred_part = nullptr;
};

namespace {

int ce_chunks(const rtx_mlp* m) { return (int)((m->C + kCeChunk - 1) / kCeChunk); }
int ce_steps(const rtx_mlp* m) { return (int)((m->C + 31) / 32); }  // 32 classes each

void mlp_free_acts(rtx_mlp* m) {
  float** bufs[] = {&m->X,  &m->H1, &m->H2,  &m->Q,      &m->dQ, &m->dH2, &m->dH1,
                    &m->pm, &m->ps, &m->lse, &m->target, &m->qa, &m->qt};
  for (float** b : bufs) {
    if (*b) (void)hipFree(*b);
    *b = nullptr;
  }
  m->cap = 0;
}

rtx_status mlp_ensure(rtx_mlp* m, uint32_t rows) {
  if (rows <= m->cap) return RTX_OK;
  mlp_free_acts(m);
  const size_t nch = (size_t)ce_chunks(m), b = ((size_t)rows + 31) / 32 * 32;
  const size_t sizes[] = {b * kInPad, b * kHid, b * kHid, b * kEmb, b * kEmb, b * kHid, b * kHid,
                          b * nch,    b * nch,  b,        b,        b * 16,   b * 16};
  float** bufs[] = {&m->X,  &m->H1, &m->H2,  &m->Q,      &m->dQ, &m->dH2, &m->dH1,
                    &m->pm, &m->ps, &m->lse, &m->target, &m->qa, &m->qt};
  for (int k = 0; k < 13; ++k)
    if (hipMalloc(bufs[k], sizes[k] * sizeof(float)) != hipSuccess) {
      (void)hipGetLastError();
      mlp_free_acts(m);
      return RTX_ERR_OUT_OF_MEMORY;
    }
  m->cap = rows;
  return RTX_OK;
}

#define MK(...)                     \
  do {                              \
    if ((__VA_ARGS__) != hipSuccess) { \
      (void)hipGetLastError();      \
      return RTX_ERR_HIP;           \
    }                               \
  } while (0)

Weights weights_of(const rtx_mlp* m) {
  return Weights{m->P + m->oW1, m->P + m->ob1, m->P + m->oW2, m->P + m->ob2, m->P + m->oW3, m->P + m->ob3};
}

// Pack the operands of a forward pass, or of a training step.
hipError_t pack(rtx_mlp* m, bool train) {
  const int count = train ? kFragEnd : kFragForward, c_tiles = train ? 2 * ce_steps(m) : 0;
  hipLaunchKernelGGL(pack_operands, dim3((count + 2 * c_tiles + 3) / 4), dim3(256), 0, m->stream, weights_of(m), count,
                     m->frags, m->P + m->oO, m->P + m->oc, (int)m->C, c_tiles, m->oa, m->ot, m->cbp);
  return hipGetLastError();
}

// Prediction: rows per pass, (row, class split) results it keeps (at most
// 10 MB), and the most workgroups it aims at (the five that a CU holds).
constexpr uint32_t kPredRows = 65536, kPredParts = 4 * kPredRows, kPredBlocks = 1280;

// Batches of at most this many rows accumulate in 64-deep partial products.
constexpr uint32_t kChunkedRows = 1984;

// Forward + backward of one batch; gradients are added into m->G, whose output
// layer is overwritten.
rtx_status mlp_fwd_bwd(rtx_mlp* m, const rtx_mlp_sample* s, uint32_t n, float inv_n) {
  hipStream_t st = m->stream;
  float *P = m->P, *G = m->G;
  uint4 *qa = reinterpret_cast<uint4*>(m->qa), *qt = reinterpret_cast<uint4*>(m->qt);
  uint32_t* target = reinterpret_cast<uint32_t*>(m->target);
  const int C = (int)m->C, nch = ce_chunks(m), c_steps = ce_steps(m), row_steps = (int)((n + 31) / 32);
  MK(pack(m, true));
  // whole 32-row steps: the tiles past n are zero queries
  hipLaunchKernelGGL(trunk_forward<true>, dim3(2 * row_steps), dim3(256), 0, st, s, (int)n, P + m->oE, (int)m->T,
                     weights_of(m), m->frags, n <= kChunkedRows ? 0 : INT_MAX, m->X, m->H1, m->H2, m->Q, qa, qt);
  hipLaunchKernelGGL(ce_stats, dim3(row_steps, (nch + 3) / 4), dim3(256), 0, st, qa, (int)n, m->oa, m->cbp, 2 * c_steps,
                     nch, m->pm, m->ps);
  hipLaunchKernelGGL(ce_finish, dim3(row_steps * 8), dim3(256), 0, st, m->pm, m->ps, nch, m->Q, P + m->oO, P + m->oc, s,
                     (int)n, C, inv_n, m->lse, target, m->loss, m->dQ);
  const int q_blocks = (c_steps + 4 * (kCeRange / 32) - 1) / (4 * (kCeRange / 32));
  const CeGrad ce{qa,   qt,        m->oa, m->ot,   m->cbp,   m->lse, target,    (int)n,
                  row_steps, C,    c_steps, q_blocks, inv_n, G + m->oO, G + m->oc, m->dQ};
  hipLaunchKernelGGL(ce_grad, dim3(c_steps + row_steps * q_blocks), dim3(256), 0, st, ce);
  hipLaunchKernelGGL(trunk_backward, dim3((n + kRowTile - 1) / kRowTile), dim3(256), 0, st, s, (int)n, (int)m->T,
                     m->frags, m->dQ, m->H1, m->H2, m->dH1, m->dH2,
                     Gradients{G + m->oE, G + m->ob1, G + m->ob2, G + m->ob3}, m->touched);
  // row ranges of at least 128 rows, at most 16
  const int ranges = std::max(1, std::min(16, (int)(n / 128)));
  const int rows_per = ((int)n + ranges - 1) / ranges;
  hipLaunchKernelGGL(weight_grads, dim3(44, ranges), dim3(256), 0, st,
                     WeightGrad{m->X, m->dH1, G + m->oW1, kInPad, kHid}, WeightGrad{m->H1, m->dH2, G + m->oW2, kHid, kHid},
                     WeightGrad{m->H2, m->dQ, G + m->oW3, kHid, kEmb}, (int)n, rows_per);
  MK(hipGetLastError());
  return RTX_OK;
}

rtx_status mlp_adam(rtx_mlp* m, float lr, bool clear) {
  m->steps++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - powf(b1, (float)m->steps), c2 = 1.f - powf(b2, (float)m->steps);
  hipLaunchKernelGGL(adam_step, dim3(2048), dim3(256), 0, m->stream, m->P, m->G, m->M1, m->V1, m->touched,
                     (size_t)m->T + 1, m->count, clear ? 1 : 0, lr, b1, b2, 1e-8f, c1, c2);
  MK(hipGetLastError());
  return RTX_OK;
}

uint64_t splitmix(uint64_t& s) {
  uint64_t z = (s += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

}  // namespace

// Context access (api.cpp).
namespace rtx_internal {
rtx_status ctx_stream(rtx_ctx* c, hipStream_t* s, int* device);
}

extern "C" {

rtx_status rtx_mlp_create(rtx_ctx* c, uint32_t n_treelets, uint32_t n_classes, uint64_t seed, rtx_mlp** out) {
  if (!c || !out || n_treelets == 0 || n_classes == 0) return RTX_ERR_INVALID_ARGUMENT;
  *out = nullptr;
  rtx_mlp* m = new (std::nothrow) rtx_mlp();
  if (!m) return RTX_ERR_OUT_OF_MEMORY;
  m->ctx = c;
  if (rtx_internal::ctx_stream(c, &m->stream, &m->device) != RTX_OK) {
    delete m;
    return RTX_ERR_INVALID_ARGUMENT;
  }
  m->T = n_treelets;
  m->C = n_classes;
  size_t o = 0;
  m->oE = o;  o += (size_t)(n_treelets + 1) * kEmb;
  m->oW1 = o; o += (size_t)kInPad * kHid;
  m->ob1 = o; o += kHid;
  m->oW2 = o; o += (size_t)kHid * kHid;
  m->ob2 = o; o += kHid;
  m->oW3 = o; o += (size_t)kHid * kEmb;
  m->ob3 = o; o += kEmb;
  m->oO = o;  o += (size_t)n_classes * kEmb;
  m->oc = o;  o += n_classes;
  m->count = o;
  (void)hipSetDevice(m->device);
  if (hipMalloc(&m->P, o * 4) != hipSuccess || hipMalloc(&m->G, o * 4) != hipSuccess ||
      hipMalloc(&m->M1, o * 4) != hipSuccess || hipMalloc(&m->V1, o * 4) != hipSuccess ||
      hipMalloc(&m->loss, 4) != hipSuccess || hipMalloc(&m->frags, kFragEnd * 1024) != hipSuccess ||
      hipMalloc(&m->oa, (size_t)ce_steps(m) * 2048) != hipSuccess ||
      hipMalloc(&m->ot, (size_t)ce_steps(m) * 2048) != hipSuccess ||
      hipMalloc(&m->cbp, (size_t)ce_steps(m) * 128) != hipSuccess ||
      hipMalloc(&m->touched, (size_t)n_treelets + 1) != hipSuccess) {
    (void)hipGetLastError();
    rtx_mlp_destroy(m);
    return RTX_ERR_OUT_OF_MEMORY;
  }
  // He-style uniform init for weights, small embeddings, zero biases.
  std::vector<float> h(o, 0.f);
  uint64_t s = seed ^ 0x6d6c70ull;
  auto uni = [&](float a) { return a * (2.f * (float)((splitmix(s) >> 40) * (1.0 / 16777216.0)) - 1.f); };
  for (size_t k = m->oE; k < m->oW1; ++k) h[k] = uni(0.5f);
  for (size_t r = 0; r < (size_t)kInPad; ++r)
    for (size_t j = 0; j < (size_t)kHid; ++j) h[m->oW1 + r * kHid + j] = r < (size_t)kIn ? uni(sqrtf(6.f / kIn)) : 0.f;
  for (size_t k = m->oW2; k < m->ob2; ++k) h[k] = uni(sqrtf(6.f / kHid));
  for (size_t k = m->oW3; k < m->ob3; ++k) h[k] = uni(sqrtf(6.f / kHid));
  for (size_t k = m->oO; k < m->oc; ++k) h[k] = uni(sqrtf(3.f / kEmb));
  if (hipMemcpy(m->P, h.data(), o * 4, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(m->G, 0, o * 4) != hipSuccess || hipMemset(m->M1, 0, o * 4) != hipSuccess ||
      hipMemset(m->V1, 0, o * 4) != hipSuccess || hipMemset(m->touched, 0, (size_t)n_treelets + 1) != hipSuccess) {
    rtx_mlp_destroy(m);
    return RTX_ERR_HIP;
  }
  *out = m;
  return RTX_OK;
}

rtx_status rtx_mlp_destroy(rtx_mlp* m) {
  if (!m) return RTX_ERR_INVALID_ARGUMENT;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  mlp_free_acts(m);
  float* bufs[] = {m->P, m->G, m->M1, m->V1, m->loss};
  for (float* b : bufs)
    if (b) (void)hipFree(b);
  void* more[] = {m->frags, m->oa, m->ot, m->cbp, m->touched};
  for (void* b : more)
    if (b) (void)hipFree(b);
  if (m->pred_q) (void)hipFree(m->pred_q);
  if (m->pred_part) (void)hipFree(m->pred_part);
  delete m;
  return RTX_OK;
}

rtx_status rtx_mlp_param_count(const rtx_mlp* m, uint64_t* count) {
  if (!m || !count) return RTX_ERR_INVALID_ARGUMENT;
  *count = m->count;
  return RTX_OK;
}

rtx_status rtx_mlp_get_params(rtx_mlp* m, float* params_host, float* grads_host) {
  if (!m) return RTX_ERR_INVALID_ARGUMENT;
  MK(hipSetDevice(m->device));
  MK(hipStreamSynchronize(m->stream));
  if (params_host) MK(hipMemcpy(params_host, m->P, m->count * 4, hipMemcpyDeviceToHost));
  if (grads_host) MK(hipMemcpy(grads_host, m->G, m->count * 4, hipMemcpyDeviceToHost));
  return RTX_OK;
}

rtx_status rtx_mlp_set_params(rtx_mlp* m, const float* params_host) {
  if (!m || !params_host) return RTX_ERR_INVALID_ARGUMENT;
  MK(hipSetDevice(m->device));
  MK(hipStreamSynchronize(m->stream));
  MK(hipMemcpy(m->P, params_host, m->count * 4, hipMemcpyHostToDevice));
  return RTX_OK;
}

rtx_status rtx_mlp_loss_grad(rtx_mlp* m, const rtx_mlp_sample* samples, uint32_t n, float* loss) {
  if (!m || !samples || n == 0) return RTX_ERR_INVALID_ARGUMENT;
  MK(hipSetDevice(m->device));
  rtx_status st = mlp_ensure(m, n);
  if (st != RTX_OK) return st;
  MK(hipMemsetAsync(m->G, 0, m->count * 4, m->stream));
  MK(hipMemsetAsync(m->loss, 0, 4, m->stream));
  st = mlp_fwd_bwd(m, samples, n, 1.f / (float)n);
  if (st != RTX_OK) return st;
  if (loss) MK(hipMemcpyAsync(loss, m->loss, 4, hipMemcpyDeviceToHost, m->stream));
  MK(hipStreamSynchronize(m->stream));
  return RTX_OK;
}

rtx_status rtx_mlp_train(rtx_mlp* m, const rtx_mlp_sample* samples, uint32_t n, uint32_t epochs, uint32_t batch,
                         float lr, float* last_epoch_loss) {
  if (!m || !samples || n == 0 || batch == 0 || epochs == 0) return RTX_ERR_INVALID_ARGUMENT;
  MK(hipSetDevice(m->device));
  batch = std::min(batch, n);
  rtx_status st = mlp_ensure(m, batch);
  if (st != RTX_OK) return st;
  float epoch_loss = 0.f;
  for (uint32_t e = 0; e < epochs; ++e) {
    MK(hipMemsetAsync(m->loss, 0, 4, m->stream));
    uint32_t nb = 0;
    if (e == 0) MK(hipMemsetAsync(m->G, 0, m->count * 4, m->stream));
    for (uint32_t b0 = 0; b0 < n; b0 += batch) {
      const uint32_t b = std::min(batch, n - b0);
      st = mlp_fwd_bwd(m, samples + b0, b, 1.f / (float)b);
      if (st != RTX_OK) return st;
      // the last batch's gradients stay readable
      st = mlp_adam(m, lr, !(e + 1 == epochs && b0 + b == n));
      if (st != RTX_OK) return st;
      ++nb;
    }
    MK(hipMemcpyAsync(&epoch_loss, m->loss, 4, hipMemcpyDeviceToHost, m->stream));
    MK(hipStreamSynchronize(m->stream));
    epoch_loss /= (float)nb;
  }
  if (last_epoch_loss) *last_epoch_loss = epoch_loss;
  return RTX_OK;
}

rtx_status rtx_mlp_predict(rtx_mlp* m, const rtx_mlp_sample* samples, uint32_t n, uint32_t* top4_dev,
                           float* probs_dev) {
  if (!m || !samples || !top4_dev || n == 0) return RTX_ERR_INVALID_ARGUMENT;
  MK(hipSetDevice(m->device));
  if (!m->pred_q) {
    // both or neither
    if (hipMalloc(&m->pred_q, (size_t)kPredRows * kEmb * 4) != hipSuccess ||
        hipMalloc(&m->pred_part, (size_t)kPredParts * sizeof(Top4)) != hipSuccess) {
      (void)hipGetLastError();
      if (m->pred_q) (void)hipFree(m->pred_q);
      m->pred_q = nullptr;
      m->pred_part = nullptr;
      return RTX_ERR_OUT_OF_MEMORY;
    }
  }
  // the last rows past a multiple of 4,096 are a batch of their own
  const uint32_t last = n % 4096;
  const uint32_t chunk_from = last && last <= kChunkedRows ? n - last : n;
  MK(pack(m, false));
  for (uint32_t b0 = 0; b0 < n; b0 += kPredRows) {
    const uint32_t b = std::min(kPredRows, n - b0);
    // class splits: enough workgroups for the chip, of whole LDS stages
    const uint32_t row_blocks = (b + 63) / 64;
    uint32_t splits = std::max(1u, std::min(kPredBlocks / row_blocks, (m->C + 2 * kCeCls - 1) / (2 * kCeCls)));
    splits = std::min(splits, std::max(1u, kPredParts / b));
    const uint32_t stages = ((m->C + kCeCls - 1) / kCeCls + splits - 1) / splits;
    const int cper = (int)(stages * kCeCls);
    splits = (m->C + cper - 1) / cper;
    hipLaunchKernelGGL(trunk_forward<false>, dim3((b + kRowTile - 1) / kRowTile), dim3(256), 0, m->stream,
                       samples + b0, (int)b, m->P + m->oE, (int)m->T, weights_of(m), m->frags,
                       chunk_from <= b0 ? 0 : (int)std::min(chunk_from - b0, b), (float*)nullptr, (float*)nullptr,
                       (float*)nullptr, m->pred_q, (uint4*)nullptr, (uint4*)nullptr);
    hipLaunchKernelGGL(logits_top4, dim3(row_blocks, splits), dim3(256), 0, m->stream, m->pred_q, (int)b,
                       m->P + m->oO, m->P + m->oc, (int)m->C, cper, m->pred_part);
    hipLaunchKernelGGL(top4_finish, dim3((b + 63) / 64), dim3(64), 0, m->stream, m->pred_part, (int)b, (int)splits,
                       top4_dev + (size_t)b0 * 4, probs_dev ? probs_dev + (size_t)b0 * 4 : nullptr);
    MK(hipGetLastError());
  }
  MK(hipStreamSynchronize(m->stream));
  return RTX_OK;
}

rtx_status rtx_mlp_gemm(rtx_ctx* c, int M, int N, int K, int trans_a, int trans_b, const float* A_dev,
                              const float* B_dev, float* C_dev) {
  hipStream_t s;
  int dev;
  if (!c || rtx_internal::ctx_stream(c, &s, &dev) != RTX_OK || M <= 0 || N <= 0 || K <= 0) return RTX_ERR_INVALID_ARGUMENT;
  MK(hipSetDevice(dev));
  const int lda = trans_a ? M : K, ldb = trans_b ? K : N;
  hipError_t e;
  if (!trans_a && !trans_b) e = gemm<false, false>(s, M, N, K, A_dev, lda, B_dev, ldb, C_dev, N, 0);
  else if (!trans_a && trans_b) e = gemm<false, true>(s, M, N, K, A_dev, lda, B_dev, ldb, C_dev, N, 0);
  else if (trans_a && !trans_b) e = gemm<true, false>(s, M, N, K, A_dev, lda, B_dev, ldb, C_dev, N, 0);
  else e = gemm<true, true>(s, M, N, K, A_dev, lda, B_dev, ldb, C_dev, N, 0);
  MK(e);
  MK(hipStreamSynchronize(s));
  return RTX_OK;
}

}  // extern "C"
