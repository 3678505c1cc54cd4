// Whole-network kernels of the screen's BF16 MLP.
//
// A layer of 256 columns on a batch of 128 is 0.1 us of MFMA work: one launch per
// GEMM, activation and update (23 for a training step of three layers) leaves
// the GPU waiting for launches.  The rows of a batch pass through the network
// independently, forward and backward, so one workgroup takes 16 rows through
// all layers, the loss and back to the first layer's pre-activations, with the
// activations in LDS; only the gradients of the weights mix rows, and a second
// launch forms them tile by tile and applies Adam where they stand.  A step is
// two launches (o16 widths 128-256-256-136, batch 128: 208 -> 38 us), the
// ensemble's prediction one, every member a grid row.
// Every element goes through the same MFMAs in the same order of k, the same
// roundings and the same scalar expressions as in mlp_kernels.hip.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include "bf16_split.h"
#include "mlp_fused.h"

namespace pamd {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

namespace {

__device__ __forceinline__ bf16x8 load8(const uint16_t *row, int k, int K, bool ok) {
  u32x4 w = {0u, 0u, 0u, 0u};
  if (ok && k < K) w = *(const u32x4 *)(row + k);
  return __builtin_bit_cast(bf16x8, w);
}
__device__ __forceinline__ float silu(float z) { return z / (1.f + __expf(-z)); }
__device__ __forceinline__ float dsilu(float z) {
  const float sg = 1.f / (1.f + __expf(-z));
  return sg * (1.f + z * (1.f - sg));
}
__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float((unsigned)b << 16); }

// one 16 x 16 tile: sum over k of a[.][k] b[.][k], in steps of 32
__device__ __forceinline__ f32x4 tile_mma(const uint16_t *a, bool aok, const uint16_t *b, bool bok, int K, int g) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int k0 = 0; k0 < K; k0 += 32) {
    const int k = k0 + 8 * g;
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load8(a, k, K, aok), load8(b, k, K, bok), acc, 0, 0, 0);
  }
  return acc;
}

}  // namespace

// LDS: hidden layer l keeps its activations, later its dZ, as bf16 [16][N + 8],
// and when training its pre-activations as float [16][N + 1]; the last layer's
// dZ likewise.
struct MlpLds {
  int act[kMlpMaxLayers], pre[kMlpMaxLayers], total;
};
__host__ __device__ inline MlpLds mlp_lds(int nl, const int *size, bool train) {
  MlpLds L;
  int off = 0;
  for (int l = 0; l < nl; ++l) {
    L.act[l] = off;
    if (l < nl - 1 || train) off += 16 * (size[l + 1] + 8) * 2;
    L.pre[l] = off;
    if (l < nl - 1 && train) off += 16 * (size[l + 1] + 1) * 4;
  }
  L.total = off;
  return L;
}

template <bool TRAIN>
__global__ __launch_bounds__(512) void k_mlp_rows(MlpNet A, MlpRows R) {
  extern __shared__ __align__(16) char lds[];
  __shared__ float red[8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.x * 16, mem = blockIdx.y, nl = A.nl;
  const bool rok = m0 + i < R.rows;
  const MlpLds L = mlp_lds(nl, A.size, TRAIN);
  float loss = 0.f;
  for (int l = 0; l < nl; ++l) {
    const int K = A.size[l], N = A.size[l + 1];
    const bool last = l == nl - 1;
    const uint16_t *a = l == 0 ? R.x + (size_t)(rok ? m0 + i : 0) * K : (const uint16_t *)(lds + L.act[l - 1]) + i * (K + 8);
    uint16_t *act = (uint16_t *)(lds + L.act[l]);
    float *pre = (float *)(lds + L.pre[l]);
    for (int tn = wave; tn * 16 < N; tn += 8) {
      const int n = tn * 16 + i;
      const bool nok = n < N;
      const f32x4 acc = tile_mma(a, l > 0 || rok, A.wb[mem][l] + (size_t)(nok ? n : 0) * K, nok, K, g);
      if (!nok) continue;
      const float bias = A.b[mem][l][n];
      unsigned pk[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 4 * g + r;
        const float z = acc[r] + bias;
        const bool ok = m0 + m < R.rows;
        if (!last) {
          if (TRAIN) pre[m * (N + 1) + n] = z;
          pk[r] = bf16_bits(silu(z));
          act[m * (N + 8) + n] = (uint16_t)pk[r];
        } else if (!TRAIN) {
          if (ok) R.out[((size_t)mem * R.rows + m0 + m) * N + n] = z;
        } else {
          float d = 0.f;
          if (ok) {
            const float e = z - R.y[(size_t)(m0 + m) * N + n];
            loss += e * e;
            d = 2.f * e / (R.rows * N);
          }
          pk[r] = bf16_bits(d);
          act[m * (N + 8) + n] = (uint16_t)pk[r];
        }
      }
      if (TRAIN && m0 + 4 * g < R.rows) {  // (rows % 8 == 0: four rows are in or out together)
        const u32x2 four = {pk[0] | (pk[1] << 16), pk[2] | (pk[3] << 16)};
        uint16_t *t = last ? R.dzt[l] : R.yt[l];
        *(u32x2 *)(t + (size_t)n * R.rows + m0 + 4 * g) = four;
      }
    }
    __syncthreads();
  }
  if (!TRAIN) return;
  for (int l = nl - 1; l > 0; --l) {
    // dZ of layer l - 1 = (dZ of layer l) W_l times the activation's derivative
    const int N = A.size[l + 1], K = A.size[l];
    const uint16_t *a = (const uint16_t *)(lds + L.act[l]) + i * (N + 8);
    uint16_t *dz = (uint16_t *)(lds + L.act[l - 1]);
    const float *pre = (const float *)(lds + L.pre[l - 1]);
    for (int tk = wave; tk * 16 < K; tk += 8) {
      const int k = tk * 16 + i;
      const bool kok = k < K;
      const f32x4 acc = tile_mma(a, true, R.wt[l] + (size_t)(kok ? k : 0) * N, kok, N, g);
      if (!kok) continue;
      unsigned pk[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 4 * g + r;
        pk[r] = bf16_bits(acc[r] * dsilu(pre[m * (K + 1) + k]));
        dz[m * (K + 8) + k] = (uint16_t)pk[r];
      }
      if (m0 + 4 * g < R.rows) {
        const u32x2 four = {pk[0] | (pk[1] << 16), pk[2] | (pk[3] << 16)};
        *(u32x2 *)(R.dzt[l - 1] + (size_t)k * R.rows + m0 + 4 * g) = four;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
  if (lane == 0) red[wave] = loss;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int w = 0; w < 8; ++w) s += red[w];
    R.part[blockIdx.x] = s;
  }
}

// Adam (decoupled weight decay) of one value
__device__ __forceinline__ float adam_one(float *w, float *m1, float *m2, size_t t, float gi, const MlpAdam &o,
                                          float wd) {
  const float a = o.b1 * m1[t] + (1.f - o.b1) * gi;
  const float b = o.b2 * m2[t] + (1.f - o.b2) * gi * gi;
  m1[t] = a;
  m2[t] = b;
  float x = w[t];
  x -= o.lr * ((a / o.c1) / (sqrtf(b / o.c2) + o.eps) + wd * x);
  w[t] = x;
  return x;
}

// Work items of a wave: the 16 x 16 tiles of every layer's dW = dZ^T X, then 64
// bias entries each, then the loss.
__global__ __launch_bounds__(256) void k_mlp_update(MlpNet A, MlpRows R, MlpAdam o) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  for (int l = 0; l < A.nl; ++l) {
    const int K = A.size[l], N = A.size[l + 1];
    const int tk = (K + 15) / 16, tiles = tk * ((N + 15) / 16);
    if (item >= tiles) {
      item -= tiles;
      continue;
    }
    const int n0 = item / tk * 16, k = item % tk * 16 + i;
    const bool nok = n0 + i < N, kok = k < K;
    const uint16_t *xt = l == 0 ? R.xt : R.yt[l - 1];
    const f32x4 acc = tile_mma(R.dzt[l] + (size_t)(nok ? n0 + i : 0) * R.rows, nok,
                               xt + (size_t)(kok ? k : 0) * R.rows, kok, R.rows, g);
    if (!kok) return;
    unsigned pk[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + 4 * g + r;
      if (n >= N) return;  // (N % 8 == 0: four rows are in or out together)
      const size_t t = (size_t)n * K + k;
      pk[r] = bf16_bits(adam_one(R.w[l], R.m_w[l], R.v_w[l], t, acc[r], o, o.wd));
      R.wb[l][t] = (uint16_t)pk[r];
    }
    const u32x2 four = {pk[0] | (pk[1] << 16), pk[2] | (pk[3] << 16)};
    *(u32x2 *)(R.wt[l] + (size_t)k * N + n0 + 4 * g) = four;
    return;
  }
  for (int l = 0; l < A.nl; ++l) {
    const int N = A.size[l + 1], blocks = (N + 63) / 64;
    if (item >= blocks) {
      item -= blocks;
      continue;
    }
    const int n = item * 64 + lane;
    if (n >= N) return;
    const uint16_t *dz = R.dzt[l] + (size_t)n * R.rows;
    float s = 0.f;
    for (int m = 0; m < R.rows; m += 8) {
      const u32x4 q = *(const u32x4 *)(dz + m);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s += bf16_to_f32((uint16_t)(q[r] & 0xffffu));
        s += bf16_to_f32((uint16_t)(q[r] >> 16));
      }
    }
    adam_one(R.bias[l], R.m_b[l], R.v_b[l], n, s, o, 0.f);
    return;
  }
  if (item != 0) return;
  const int np = (R.rows + 15) / 16;
  float s = 0.f;
  for (int p = lane; p < np; p += 64) s += R.part[p];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) *R.loss = s / (R.rows * A.size[A.nl]);
}

// out[row][p] = bf16((x[row][p] - mean[p]) / std[p]) for p < n, 0 up to ld
__global__ void k_standardise(int rows, int n, int ld, const double *x, const double *mean, const double *std_,
                              uint16_t *out) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)rows * ld) return;
  const int p = (int)(t % ld);
  const size_t row = t / ld;
  unsigned b = 0;
  if (p < n) b = bf16_bits((float)((x[row * n + p] - mean[p]) / std_[p]));
  out[t] = (uint16_t)b;
}

int mlp_lds_bytes(int nl, const int *size, bool train) { return mlp_lds(nl, size, train).total; }

hipError_t launch_mlp_forward(const MlpNet &a, const MlpRows &r, int members, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_rows<false>, dim3((r.rows + 15) / 16, members), dim3(512),
                     mlp_lds_bytes(a.nl, a.size, false), s, a, r);
  return hipGetLastError();
}

hipError_t launch_mlp_train(const MlpNet &a, const MlpRows &r, const MlpAdam &o, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_rows<true>, dim3((r.rows + 15) / 16), dim3(512), mlp_lds_bytes(a.nl, a.size, true), s,
                     a, r);
  int items = 1;
  for (int l = 0; l < a.nl; ++l)
    items += (a.size[l] + 15) / 16 * ((a.size[l + 1] + 15) / 16) + (a.size[l + 1] + 63) / 64;
  hipLaunchKernelGGL(k_mlp_update, dim3((items + 3) / 4), dim3(256), 0, s, a, r, o);
  return hipGetLastError();
}

hipError_t launch_standardise(int rows, int n, int ld, const double *x, const double *mean, const double *std_,
                              uint16_t *out, hipStream_t s) {
  const size_t total = (size_t)rows * ld;
  hipLaunchKernelGGL(k_standardise, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, rows, n, ld, x, mean,
                     std_, out);
  return hipGetLastError();
}

}  // namespace pamd
