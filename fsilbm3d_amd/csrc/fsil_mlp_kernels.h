// Learned warm start of the multi-direct-forcing loop: a 12 -> 64 -> 64 -> 64
// -> 3 perceptron (tanh hidden layers) per immersed-boundary marker.
//
// Training runs in FP32 on the matrix cores (k_mlp_rows: forward, backward and
// weight gradients in one launch; k_mlp_reduce: the sums and Adam), every sum
// in a fixed order so a run is reproducible.  Inference runs on the
// matrix cores: BF16 operands, FP32 accumulation (v_mfma_f32_16x16x16_bf16),
// one wave per 16 markers, the weights of all layers held in LDS as BF16.
//
// Parameter layout (floats): W1[64][12] b1[64] W2[64][64] b2[64] W3[64][64]
// b3[64] W4[3][64] b4[3]; W[o][i] multiplies input i into output o.
#pragma once
#include <type_traits>

#include "fsil_common.h"

namespace fsil {

constexpr int kMlpIn = 12, kMlpH = 64, kMlpOut = 3;
constexpr int kMlpOffW1 = 0, kMlpOffB1 = kMlpOffW1 + kMlpH * kMlpIn;
constexpr int kMlpOffW2 = kMlpOffB1 + kMlpH, kMlpOffB2 = kMlpOffW2 + kMlpH * kMlpH;
constexpr int kMlpOffW3 = kMlpOffB2 + kMlpH, kMlpOffB3 = kMlpOffW3 + kMlpH * kMlpH;
constexpr int kMlpOffW4 = kMlpOffB3 + kMlpH, kMlpOffB4 = kMlpOffW4 + kMlpOut * kMlpH;
constexpr int kMlpParams = kMlpOffB4 + kMlpOut;

// ---------------------------------------------------------------------------
// FP32 training kernels (matrix cores, FP32 operands)

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One pass over the rows for the whole network: forward, loss and backward of
// 64-row tiles with the weights and the tile's activations in LDS, the weight
// gradients accumulated in registers over a workgroup's tiles.  All products
// are v_mfma_f32_16x16x4_f32 (FP32 operands and sums).
//
// Bound: the FP32 matrix cores (3 x 9.3k multiply-adds per row), at the sizes
// in use the launch and the host copies.  One thread per weight walking all
// the rows, a launch per layer, took 8.6 ms per layer at 36,864 rows (34.9 ms
// in all) where this kernel takes 54 us (38 TFLOP/s).
//
// Eight waves: wave w holds rows (w & 3) * 16.. of the tile and columns
// (w >> 2) * 32.. (two 16x16 results) of each product.  LDS row strides of 84
// (activations, weights) and 20 words (inputs) put both operand reads, 16
// rows x 4 columns and 4 rows x 16 columns, on (nearly) distinct banks.
constexpr int kGradThreads = 512, kGradRows = 64, kGradBlocks = 256;
constexpr int kLdH = 84, kLdX = 20;

struct MlpGradLds {
  float w1[64 * kLdX], w2[64 * kLdH], w3[64 * kLdH], w4[16 * kLdH];
  float b1[64], b2[64], b3[64], b4[16];
  float x[kGradRows * kLdX], dy[kGradRows * kLdX];
  float h1[kGradRows * kLdH], h2[kGradRows * kLdH], h3[kGradRows * kLdH];
  double e2[kGradThreads / 64];
};

// c + A B over KS steps of 4: lane l takes A[l % 16][4 ks + l / 16] and
// B[4 ks + l / 16][l % 16]; the result is C[4 (l / 16) + r][l % 16].  (sa, ka)
// and (sb, kb): strides of A's row and step index, of B's column and step index.
template <int KS>
__device__ __forceinline__ f32x4 mfma_f32(const float *A, int sa, int ka, const float *B, int sb, int kb, f32x4 c) {
  const int l = threadIdx.x & 63, i = l & 15, q = l >> 4;
  A += i * sa + q * ka;
  B += i * sb + q * kb;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(A[4 * ks * ka], B[4 * ks * kb], c, 0, 0, 0);
  return c;
}
// the same with B all ones: every column holds A's row sums
template <int KS>
__device__ __forceinline__ f32x4 mfma_f32_ones(const float *A, int sa, int ka, f32x4 c) {
  const int l = threadIdx.x & 63;
  A += (l & 15) * sa + (l >> 4) * ka;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) c = __builtin_amdgcn_mfma_f32_16x16x4f32(A[4 * ks * ka], 1.0f, c, 0, 0, 0);
  return c;
}

// Rows idx[0..n) (idx null: 0..n) of X and Yt.  GRAD: the gradient of the mean
// squared error over the n x 3 outputs, this workgroup's part into gpart
// (kMlpParams per workgroup) and its squared errors into epart; else the
// outputs into Yp.
template <bool GRAD>
__global__ __launch_bounds__(kGradThreads) void k_mlp_rows(const float *__restrict__ X, const float *__restrict__ Yt,
                                                           const int *__restrict__ idx, int n,
                                                           const float *__restrict__ th, float *__restrict__ Yp,
                                                           float *__restrict__ gpart, double *__restrict__ epart) {
  extern __shared__ __align__(16) char mlp_lds_raw[];
  MlpGradLds &L = *reinterpret_cast<MlpGradLds *>(mlp_lds_raw);
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, i16 = l & 15, q4 = (l >> 4) * 4;
  const int rs = (w & 3) * 16, ch = (w >> 2) * 32;
  for (int i = tid; i < 64 * kLdX; i += kGradThreads) {
    const int o = i / kLdX, k = i - o * kLdX;
    L.w1[i] = k < kMlpIn ? th[kMlpOffW1 + o * kMlpIn + k] : 0.0f;
  }
  for (int i = tid; i < 64 * 64; i += kGradThreads) {
    const int o = i >> 6, k = i & 63;
    L.w2[o * kLdH + k] = th[kMlpOffW2 + i];
    L.w3[o * kLdH + k] = th[kMlpOffW3 + i];
  }
  for (int i = tid; i < 16 * 64; i += kGradThreads) {
    const int o = i >> 6, k = i & 63;
    L.w4[o * kLdH + k] = o < kMlpOut ? th[kMlpOffW4 + i] : 0.0f;
  }
  if (tid < 64) {
    L.b1[tid] = th[kMlpOffB1 + tid];
    L.b2[tid] = th[kMlpOffB2 + tid];
    L.b3[tid] = th[kMlpOffB3 + tid];
    if (tid < 16) L.b4[tid] = tid < kMlpOut ? th[kMlpOffB4 + tid] : 0.0f;
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // weight gradients: wave w holds outputs rs.. and inputs ch.., ch + 16.. of
  // W2 and W3 (and their biases when ch == 0); waves 0-3 outputs rs.. of W1
  // and b1, waves 4-7 inputs rs.. of W4 (wave 4 also b4)
  f32x4 g2[2] = {zero, zero}, g3[2] = {zero, zero}, gb2 = zero, gb3 = zero, g14 = zero, gb14 = zero;
  double e2 = 0.0;
  const float inv = 2.0f;
  const float count = (float)(n * kMlpOut);
  const int ntile = (n + kGradRows - 1) / kGradRows;
  for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const int s0 = tile * kGradRows;
    __syncthreads();  // (the previous tile is done with x, dy, h1)
    for (int i = tid; i < kGradRows * kLdX; i += kGradThreads) {
      const int r = i / kLdX, k = i - r * kLdX, s = s0 + r;
      float v = 0.0f;
      if (s < n && k < kMlpIn) v = X[(size_t)(idx ? idx[s] : s) * kMlpIn + k];
      L.x[i] = v;
      if (GRAD) L.dy[i] = 0.0f;
    }
    __syncthreads();
    auto layer = [&](const float *A, int lda, const float *W, const float *b, float *H, auto steps) {
      constexpr int KS = decltype(steps)::value;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int c0 = ch + 16 * t;
        const float bv = b[c0 + i16];
        f32x4 c = {bv, bv, bv, bv};
        c = mfma_f32<KS>(A + rs * lda, lda, 1, W + c0 * lda, lda, 1, c);
#pragma unroll
        for (int r = 0; r < 4; ++r) H[(rs + q4 + r) * kLdH + c0 + i16] = tanhf(c[r]);
      }
      __syncthreads();
    };
    layer(L.x, kLdX, L.w1, L.b1, L.h1, std::integral_constant<int, 3>());
    layer(L.h1, kLdH, L.w2, L.b2, L.h2, std::integral_constant<int, 16>());
    layer(L.h2, kLdH, L.w3, L.b3, L.h3, std::integral_constant<int, 16>());
    if (w < 4) {  // the three outputs: columns 0..2 of one 16x16 result per row strip
      const float bv = L.b4[i16];
      f32x4 c = {bv, bv, bv, bv};
      c = mfma_f32<16>(L.h3 + rs * kLdH, kLdH, 1, L.w4, kLdH, 1, c);
      if (i16 < kMlpOut)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int s = s0 + rs + q4 + r;
          if (s < n) {
            if constexpr (GRAD) {
              const float d = c[r] - Yt[(size_t)(idx ? idx[s] : s) * kMlpOut + i16];
              L.dy[(rs + q4 + r) * kLdX + i16] = inv * d / count;
              e2 = e2 + (double)d * (double)d;
            } else {
              Yp[(size_t)s * kMlpOut + i16] = c[r];
            }
          }
        }
    }
    if constexpr (GRAD) {
      __syncthreads();
      // dZ = (dY W) (1 - H^2) of one layer, two results per wave, into d
      float d[2][4];
      auto back = [&](const float *dZ, int ldz, const float *W, const float *H, auto steps) {
        constexpr int KS = decltype(steps)::value;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int c0 = ch + 16 * t;
          const f32x4 c = mfma_f32<KS>(dZ + rs * ldz, ldz, 1, W + c0, 1, kLdH, zero);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float h = H[(rs + q4 + r) * kLdH + c0 + i16];
            d[t][r] = c[r] * (1.0f - h * h);
          }
        }
      };
      auto keep = [&](float *H) {  // d over the activations it came from
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) H[(rs + q4 + r) * kLdH + ch + 16 * t + i16] = d[t][r];
        __syncthreads();
      };
      auto wgrad = [&](const float *dZ, const float *H, f32x4 (&g)[2], f32x4 &gb) {
#pragma unroll
        for (int t = 0; t < 2; ++t) g[t] = mfma_f32<16>(dZ + rs, 1, kLdH, H + ch + 16 * t, 1, kLdH, g[t]);
        if (ch == 0) gb = mfma_f32_ones<16>(dZ + rs, 1, kLdH, gb);
      };
      back(L.dy, kLdX, L.w4, L.h3, std::integral_constant<int, 1>());
      if (w >= 4) {
        g14 = mfma_f32<16>(L.dy, 1, kLdX, L.h3 + rs, 1, kLdH, g14);
        if (w == 4) gb14 = mfma_f32_ones<16>(L.dy, 1, kLdX, gb14);
      }
      keep(L.h3);
      back(L.h3, kLdH, L.w3, L.h2, std::integral_constant<int, 16>());
      wgrad(L.h3, L.h2, g3, gb3);
      keep(L.h2);
      back(L.h2, kLdH, L.w2, L.h1, std::integral_constant<int, 16>());
      wgrad(L.h2, L.h1, g2, gb2);
      keep(L.h1);
      if (w < 4) {
        g14 = mfma_f32<16>(L.h1 + rs, 1, kLdH, L.x, 1, kLdX, g14);
        gb14 = mfma_f32_ones<16>(L.h1 + rs, 1, kLdH, gb14);
      }
    }
  }
  if constexpr (GRAD) {
    float *g = gpart + (size_t)blockIdx.x * kMlpParams;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int o = rs + q4 + r;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        g[kMlpOffW2 + o * kMlpH + ch + 16 * t + i16] = g2[t][r];
        g[kMlpOffW3 + o * kMlpH + ch + 16 * t + i16] = g3[t][r];
      }
      if (ch == 0 && i16 == 0) {
        g[kMlpOffB2 + o] = gb2[r];
        g[kMlpOffB3 + o] = gb3[r];
      }
      if (w < 4) {
        if (i16 < kMlpIn) g[kMlpOffW1 + o * kMlpIn + i16] = g14[r];
        if (i16 == 0) g[kMlpOffB1 + o] = gb14[r];
      } else if (q4 + r < kMlpOut) {
        g[kMlpOffW4 + (q4 + r) * kMlpH + rs + i16] = g14[r];
        if (w == 4 && i16 == 0) g[kMlpOffB4 + q4 + r] = gb14[r];
      }
    }
    for (int off = 32; off > 0; off >>= 1) e2 = e2 + __shfl_down(e2, off, 64);
    if (l == 0) L.e2[w] = e2;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
      for (int k = 0; k < kGradThreads / 64; ++k) t = t + L.e2[k];
      epart[blockIdx.x] = t;
    }
  }
}

// The workgroups' gradient parts added in a fixed order (four runs of them
// side by side, then the runs in order) into g, and with ADAM one step of
// Adam (Kingma & Ba 2015, algorithm 1; bc1 = 1 - beta1^t, bc2 = 1 - beta2^t)
// on the parameters.  64 parameters per workgroup.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_mlp_reduce(const float *__restrict__ gpart, int nblk, float *__restrict__ g,
                                                    float *__restrict__ th, float *__restrict__ m,
                                                    float *__restrict__ v, float lr, float b1, float b2, float eps,
                                                    float bc1, float bc2) {
  __shared__ float run[4][64];
  const int l = threadIdx.x & 63, k = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + l;
  const int per = (nblk + 3) / 4, j1 = min(nblk, (k + 1) * per);
  float s = 0.0f;
  if (i < kMlpParams)
#pragma unroll 8
    for (int j = k * per; j < j1; ++j) s = s + gpart[(size_t)j * kMlpParams + i];
  run[k][l] = s;
  __syncthreads();
  if (k || i >= kMlpParams) return;
  const float gi = ((run[0][l] + run[1][l]) + run[2][l]) + run[3][l];
  g[i] = gi;
  if constexpr (ADAM) {
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    th[i] = th[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  }
}

// ---------------------------------------------------------------------------
// BF16 matrix-core inference

typedef short bf16x4 __attribute__((ext_vector_type(4)));
// round-to-nearest-even float -> bfloat16 bits (finite inputs)
__device__ __forceinline__ short f2bf(float x) {
  unsigned u = __float_as_uint(x);
  u = u + 0x7fffu + ((u >> 16) & 1u);
  return (short)(u >> 16);
}

// LDS image of the network: BF16 weights padded to 16-multiples (W1: 64 x 16,
// W2, W3: 64 x 64, W4: 16 x 64), FP32 biases (b4 padded to 16).  Rows are
// padded by 8 bytes so that the 8-byte operand reads of 16 rows fall on
// distinct banks (rows of 128 bytes put all 16 on one).
constexpr int kLdW1 = 20, kLdW = 68;
struct MlpLds {
  short w1[64 * kLdW1];
  short w2[64 * kLdW];
  short w3[64 * kLdW];
  short w4[16 * kLdW];
  float b1[64], b2[64], b3[64], b4[16];
  short act[4][16 * kLdW];  // per wave: 16 markers x 64 activations
};

// One wave: C(16 x 16 tile nt) = A(16 x K) * W^T, A from LDS rows (K = 16*kt),
// W rows nt*16..nt*16+15 from LDS, both BF16.  Lane l holds A[l%16][4*(l/16)+j]
// and B[4*(l/16)+j][l%16] = W[l%16][4*(l/16)+j]; the result C[4*(l/16)+j][l%16].
__device__ __forceinline__ f32x4 mfma_tile(const short *A, int lda, const short *W, int ldw, int ksteps, int nt) {
  const int l = threadIdx.x & 63;
  const int r = l & 15, kq = (l >> 4) * 4;
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < ksteps; ++ks) {
    const bf16x4 a = *reinterpret_cast<const bf16x4 *>(&A[r * lda + ks * 16 + kq]);
    const bf16x4 b = *reinterpret_cast<const bf16x4 *>(&W[(nt * 16 + r) * ldw + ks * 16 + kq]);
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
  return c;
}

// Y[m][0..2] for n markers, X[m][0..11] inputs; one wave per 16 markers, each
// workgroup taking every gridDim-th 64 of them so that the weights are read
// and rounded once per workgroup (kInferBlocks of them at most: 36,864
// markers take 21.3 us; with a workgroup for every 64, and their activations
// on one bank, they took 33.9).
constexpr int kInferBlocks = 512;
__global__ __launch_bounds__(256) void k_mlp_infer_bf16(const float *__restrict__ X, int n,
                                                        const float *__restrict__ th, float *__restrict__ Y) {
  __shared__ __align__(16) MlpLds L;
  const int tid = threadIdx.x;
  // weights -> LDS (BF16), zero padding
  for (int i = tid; i < 64 * 16; i += blockDim.x) {
    const int o = i / 16, k = i % 16;
    L.w1[o * kLdW1 + k] = k < kMlpIn ? f2bf(th[kMlpOffW1 + o * kMlpIn + k]) : (short)0;
  }
  for (int i = tid; i < 64 * 64; i += blockDim.x) {
    const int o = i >> 6, k = i & 63;
    L.w2[o * kLdW + k] = f2bf(th[kMlpOffW2 + i]);
    L.w3[o * kLdW + k] = f2bf(th[kMlpOffW3 + i]);
  }
  for (int i = tid; i < 16 * 64; i += blockDim.x) {
    const int o = i / 64, k = i % 64;
    L.w4[o * kLdW + k] = o < kMlpOut ? f2bf(th[kMlpOffW4 + i]) : (short)0;
  }
  for (int i = tid; i < 64; i += blockDim.x) {
    L.b1[i] = th[kMlpOffB1 + i];
    L.b2[i] = th[kMlpOffB2 + i];
    L.b3[i] = th[kMlpOffB3 + i];
  }
  for (int i = tid; i < 16; i += blockDim.x) L.b4[i] = i < kMlpOut ? th[kMlpOffB4 + i] : 0.f;
  __syncthreads();
  // from here on each wave works on its own rows of act
  const int w = tid >> 6, l = tid & 63;
  short *act = L.act[w];
  const int col = l & 15, rq = (l >> 4) * 4;
  for (int m0 = (blockIdx.x * 4 + w) * 16; m0 < n; m0 += gridDim.x * 64) {
    // inputs -> LDS rows (16 x 16, K padded)
    for (int i = l; i < 16 * 16; i += 64) {
      const int r = i / 16, k = i % 16;
      const int m = m0 + r;
      act[r * kLdW + k] = (m < n && k < kMlpIn) ? f2bf(X[(size_t)m * kMlpIn + k]) : (short)0;
    }
    wave_sync();
    // layer 1: K = 16; layers 2 and 3: K = 64
    f32x4 c[4];
    auto finish = [&](const float *bl) {
      wave_sync();
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          act[(rq + j) * kLdW + nt * 16 + col] = f2bf(tanhf(c[nt][j] + bl[nt * 16 + col]));
      wave_sync();
    };
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) c[nt] = mfma_tile(act, kLdW, L.w1, kLdW1, 1, nt);
    finish(L.b1);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) c[nt] = mfma_tile(act, kLdW, L.w2, kLdW, 4, nt);
    finish(L.b2);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) c[nt] = mfma_tile(act, kLdW, L.w3, kLdW, 4, nt);
    finish(L.b3);
    // output layer: N = 16 (3 used)
    const f32x4 c4 = mfma_tile(act, kLdW, L.w4, kLdW, 4, 0);
    if (col < kMlpOut)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int m = m0 + rq + j;
        if (m < n) Y[(size_t)m * kMlpOut + col] = c4[j] + L.b4[col];
      }
    wave_sync();
  }
}

}  // namespace fsil
