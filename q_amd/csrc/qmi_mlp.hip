// Overlap predictor of the learned lambda schedule: a small MLP trained and
// evaluated on the GPU by the kernels in this file (no reference
// counterpart; the reference schedules lambda windows by hand).
//
//   x[n_in] -> Linear(H) -> SiLU -> Linear(H) -> SiLU -> Linear(1) -> sigmoid
//
// Weights are kept in BF16 for the forward and backward passes, with an FP32
// master copy for the optimiser (Adam); every product is accumulated in FP32.
// Networks of at most 128 inputs and 128 hidden units (the shipped one has 34
// and 128) run fused: k_mlp takes 16 rows through the whole forward and, for a
// gradient, backward pass on the FP32 matrix cores, and k_mlp_reduce sums the
// blocks' gradients and applies Adam.  Larger networks run layer by layer with
// an LDS-tiled product (k_gemm).  Reductions run in a fixed order: results are
// reproducible run to run.
#include <hip/hip_bfloat16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "../../include/qmi.h"

namespace {

thread_local std::string g_mlp_err;
int mlp_err(int code, const std::string& m) {
  g_mlp_err = m;
  return code;
}
#define MLP_OK(call)                                                                                  \
  do {                                                                                                \
    hipError_t e_ = (call);                                                                           \
    if (e_ != hipSuccess) return mlp_err(-100, std::string("HIP error: ") + hipGetErrorString(e_)); \
  } while (0)

// C[M x N] = alpha * op(A) * op(B) + beta * C, op(A) is M x K, op(B) is K x N.
// A and B are row-major FP32 or BF16 (TA / TB = 1: stored transposed).
template <typename TA_, typename TB_, bool TA, bool TB>
__global__ void __launch_bounds__(256) k_gemm(int M, int N, int K, float alpha, const TA_* A, int lda, const TB_* B,
                                              int ldb, float beta, float* C, int ldc) {
  __shared__ float sa[16][17];
  __shared__ float sb[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int row = blockIdx.y * 16 + ty, col = blockIdx.x * 16 + tx;
  float acc = 0.f;
  for (int k0 = 0; k0 < K; k0 += 16) {
    // A tile: rows blockIdx.y*16 + ty, columns k0 + tx
    {
      const int r = blockIdx.y * 16 + ty, c = k0 + tx;
      float v = 0.f;
      if (r < M && c < K) v = TA ? (float)A[(size_t)c * lda + r] : (float)A[(size_t)r * lda + c];
      sa[ty][tx] = v;
    }
    // B tile: rows k0 + ty, columns blockIdx.x*16 + tx
    {
      const int r = k0 + ty, c = blockIdx.x * 16 + tx;
      float v = 0.f;
      if (r < K && c < N) v = TB ? (float)B[(size_t)c * ldb + r] : (float)B[(size_t)r * ldb + c];
      sb[ty][tx] = v;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) acc = fmaf(sa[ty][k], sb[k][tx], acc);
    __syncthreads();
  }
  if (row < M && col < N) {
    float* c = &C[(size_t)row * ldc + col];
    *c = alpha * acc + (beta != 0.f ? beta * *c : 0.f);
  }
}

// z (B x H) += bias; a = silu(z)
__global__ void k_bias_silu(int B, int H, float* z, const float* bias, float* a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= B * H) return;
  const float v = z[i] + bias[i % H];
  z[i] = v;
  a[i] = v / (1.f + expf(-v));
}

// output layer: y = sigmoid(z3 + b3); loss terms and dz3 for MSE
__global__ void k_out(int B, float* z3, const float* b3, float* y, const float* t, float* dz3, float* lossv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= B) return;
  const float v = z3[i] + b3[0];
  z3[i] = v;
  const float s = 1.f / (1.f + expf(-v));
  y[i] = s;
  if (t) {
    const float e = s - t[i];
    lossv[i] = e * e;
    dz3[i] = 2.f * e / (float)B * s * (1.f - s);
  }
}

// dz = da * silu'(z), silu'(z) = s (1 + z (1 - s)), s = sigmoid(z)
__global__ void k_silu_back(int n, const float* z, const float* da, float* dz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float s = 1.f / (1.f + expf(-z[i]));
  dz[i] = da[i] * s * (1.f + z[i] * (1.f - s));
}

// column sums of dz (B x H) -> db (H), fixed order: a block takes 64 columns,
// its 16 row groups sum every 16th row each and are added in group order
constexpr int kSumGroups = 16;
__global__ void __launch_bounds__(64 * kSumGroups) k_colsum(int B, int H, const float* dz, float* db) {
  __shared__ float s_part[kSumGroups][64];
  const int c = threadIdx.x & 63, r = threadIdx.x >> 6, h = blockIdx.x * 64 + c;
  float s = 0.f;
  if (h < H)
    for (int b = r; b < B; b += kSumGroups) s += dz[(size_t)b * H + h];
  s_part[r][c] = s;
  __syncthreads();
  if (r != 0 || h >= H) return;
  for (int k = 1; k < kSumGroups; ++k) s += s_part[k][c];
  db[h] = s;
}

// sum of per-sample squared errors, one block, fixed order
__global__ void k_sum(int n, const float* v, float* out) {
  __shared__ float red[256];
  float s = 0.f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) s += v[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// ------------------------------------------------------ fused network --
// Packed BF16 weights of a fused network, zero where padded: W1 [kHp][ip],
// W2 [kHp][kHp] and its transpose, ip = 64 or 128 inputs.
constexpr int kHp = 128;             // hidden units of a fused network, padded
constexpr int kTileRows = 16;        // batch rows of a block's tile
constexpr int kFusedBlock = 512;     // 8 waves, one 16-column tile of the hidden layers each
constexpr int kPartBlocks = 256;     // most blocks (partial gradients) of a gradient pass
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct Net {
  int I, H;                          // inputs, hidden units
  const unsigned short *w1, *w2, *w2t;
  const hip_bfloat16* w3;
  const float *b1, *b2, *b3;         // FP32 master biases
};

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float bf_lo(unsigned u) { return __builtin_bit_cast(float, u << 16); }
__device__ __forceinline__ float bf_hi(unsigned u) { return __builtin_bit_cast(float, u & 0xffff0000u); }

// C[16 x 16] = A[16 x K] W[16 x K]^T, A in LDS (row stride ld), W packed BF16.
// A step's four k values are K/4 apart, so a lane's k values are contiguous
// and both operands load as 16-byte vectors (the sum over k takes any order).
template <int K>
__device__ __forceinline__ f32x4 tile_product(const float* A, int ld, const unsigned short* W) {
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const float* a = A + r * ld + q * (K / 4);
  const uint4* w = reinterpret_cast<const uint4*>(W + r * K + q * (K / 4));
  uint4 u[K / 32];
#pragma unroll
  for (int c = 0; c < K / 32; ++c) u[c] = w[c];
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < K / 32; ++c) {
    const f32x4 x0 = *reinterpret_cast<const f32x4*>(a + 8 * c), x1 = *reinterpret_cast<const f32x4*>(a + 8 * c + 4);
    acc = mfma4(x0[0], bf_lo(u[c].x), acc);
    acc = mfma4(x0[1], bf_hi(u[c].x), acc);
    acc = mfma4(x0[2], bf_lo(u[c].y), acc);
    acc = mfma4(x0[3], bf_hi(u[c].y), acc);
    acc = mfma4(x1[0], bf_lo(u[c].z), acc);
    acc = mfma4(x1[1], bf_hi(u[c].z), acc);
    acc = mfma4(x1[2], bf_lo(u[c].w), acc);
    acc = mfma4(x1[3], bf_hi(u[c].w), acc);
  }
  return acc;
}

// silu'(z) = s (1 + z (1 - s)), s = sigmoid(z)
__device__ __forceinline__ float silu_d(float z) {
  const float s = 1.f / (1.f + expf(-z));
  return s * (1.f + z * (1.f - s));
}

// Forward pass of B rows (row b of the batch is row idx[b] of X and T, or b
// without idx) and, with BACK, the gradient of the mean squared error: block
// k takes the 16-row tiles k, k + gridDim.x, ... and stores its sum of the
// gradient (parameter order, then its sum of squared errors) at part[k].  In
// a 16 x 16 product lane l holds column l % 16, rows 4 (l / 16) .. + 3; wave
// w owns hidden units 16 w .. 16 w + 15 of both layers, so z and dz stay in
// registers and only a1, dz2 and dz1 pass through LDS.
//
// Bound by latency: a tile is 0.5 MFLOP per layer product (32 dependent
// matrix steps), and what the layer-by-layer form spent was its 20 launches
// and the column sums' one thread per column.  16 rows per tile: a minibatch
// of 256 fills 16 CUs, where 32-row tiles would leave 8.  Measured with 34
// inputs and 128 hidden units, layer by layer before and fused now: forward of
// 777 device rows 20.6 -> 4.5 us; gradient of 7960 host rows 5127 -> 142 us;
// 8 training minibatches of 256 rows 1816 -> 251 us.
template <int IP, bool BACK>
__global__ void __launch_bounds__(kFusedBlock) k_mlp(int B, Net N, const float* __restrict__ X,
                                                     const float* __restrict__ T, const int* __restrict__ idx,
                                                     float* __restrict__ y, float* __restrict__ part) {
  constexpr int LX = IP + 4, LH = kHp + 4;   // row strides: 16-byte aligned, rows 4 banks apart
  __shared__ __align__(16) float s_x[kTileRows][LX], s_a[kTileRows][LH], s_d[BACK ? kTileRows : 1][LH];
  __shared__ float s_z3[kFusedBlock / 64][kTileRows], s_dz3[kTileRows], s_e[kTileRows];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int h = wv * 16 + c;
  const bool on = h < N.H;
  const float b1 = on ? N.b1[h] : 0.f, b2 = on ? N.b2[h] : 0.f, w3 = on ? (float)N.w3[h] : 0.f, b3 = N.b3[0];
  const unsigned short* w1 = N.w1 + (size_t)wv * 16 * IP;
  const unsigned short* w2 = N.w2 + (size_t)wv * 16 * kHp;
  const unsigned short* w2t = N.w2t + (size_t)wv * 16 * kHp;
  f32x4 g2[BACK ? kHp / 16 : 1] = {}, g1[BACK ? IP / 16 : 1] = {};   // rows h, columns by 16
  float gb1 = 0.f, gb2 = 0.f, gw3 = 0.f, gb3 = 0.f, gl = 0.f;
  const int ntile = (B + kTileRows - 1) / kTileRows;
  for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const int r0 = tile * kTileRows;
    for (int k = threadIdx.x; k < kTileRows * IP; k += kFusedBlock) {
      const int r = k / IP, i = k % IP, b = r0 + r;
      s_x[r][i] = b < B && i < N.I ? X[(size_t)(idx ? idx[b] : b) * N.I + i] : 0.f;
    }
    __syncthreads();
    f32x4 z1 = tile_product<IP>(&s_x[0][0], LX, w1);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      z1[k] += b1;
      s_a[4 * q + k][h] = on ? z1[k] / (1.f + expf(-z1[k])) : 0.f;   // padding stays 0 for any input
    }
    __syncthreads();
    f32x4 z2 = tile_product<kHp>(&s_a[0][0], LH, w2);
    f32x4 a2, p3;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      z2[k] += b2;
      a2[k] = z2[k] / (1.f + expf(-z2[k]));
      p3[k] = on ? a2[k] * w3 : 0.f;
    }
    // output unit: columns of the wave, then the waves in order
#pragma unroll
    for (int m = 8; m > 0; m >>= 1)
#pragma unroll
      for (int k = 0; k < 4; ++k) p3[k] += __shfl_xor(p3[k], m);
    if (c == 0)
      for (int k = 0; k < 4; ++k) s_z3[wv][4 * q + k] = p3[k];
    __syncthreads();
    if (threadIdx.x < kTileRows) {
      const int b = r0 + threadIdx.x;
      float z3 = b3;
      for (int k = 0; k < kFusedBlock / 64; ++k) z3 += s_z3[k][threadIdx.x];
      const float s = 1.f / (1.f + expf(-z3));
      if (b < B && y) y[b] = s;
      if (BACK) {
        const float e = b < B ? s - T[idx ? idx[b] : b] : 0.f;
        s_e[threadIdx.x] = e * e;
        s_dz3[threadIdx.x] = 2.f * e / (float)B * s * (1.f - s);
      }
    }
    if constexpr (BACK) {
      __syncthreads();
      f32x4 d2;
      float t3 = 0.f, t2 = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float d3 = s_dz3[4 * q + k];
        d2[k] = on ? d3 * w3 * silu_d(z2[k]) : 0.f;
        s_d[4 * q + k][h] = d2[k];
        t3 += d3 * a2[k];
        t2 += d2[k];
      }
      gw3 += t3;
      gb2 += t2;
      if (threadIdx.x < kTileRows) {
        gb3 += s_dz3[threadIdx.x];
        gl += s_e[threadIdx.x];
      }
      __syncthreads();
      const f32x4 d1a = tile_product<kHp>(&s_d[0][0], LH, w2t);   // dz2 W2
      // dz2^T a1: rows h of the wave's tile, one 16-column tile of a1 at a time
      float dr[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) dr[m] = s_d[4 * m + q][h];
#pragma unroll
      for (int n = 0; n < kHp / 16; ++n)
#pragma unroll
        for (int m = 0; m < 4; ++m) g2[n] = mfma4(dr[m], s_a[4 * m + q][16 * n + c], g2[n]);
      __syncthreads();
      float t1 = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float d1 = d1a[k] * silu_d(z1[k]);
        s_d[4 * q + k][h] = d1;   // the wave's own columns, which its other lanes read below
        t1 += d1;
      }
      gb1 += t1;
      // (a wave's LDS accesses are in order; the fence keeps the compiler from
      // moving the loads before the other lanes' stores, which a wave barrier
      // alone does not promise)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int m = 0; m < 4; ++m) dr[m] = s_d[4 * m + q][h];
#pragma unroll
      for (int n = 0; n < IP / 16; ++n)
#pragma unroll
        for (int m = 0; m < 4; ++m) g1[n] = mfma4(dr[m], s_x[4 * m + q][16 * n + c], g1[n]);
    }
    __syncthreads();   // the next tile overwrites the rows
  }
  if constexpr (BACK) {
    const int I = N.I, H = N.H, np = H * I + H * H + 3 * H + 1;
    float* P = part + (size_t)blockIdx.x * (np + 1);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int hr = wv * 16 + 4 * q + k;   // row of the accumulators' lane values
      if (hr >= H) continue;
#pragma unroll
      for (int n = 0; n < IP / 16; ++n)
        if (16 * n + c < I) P[hr * I + 16 * n + c] = g1[n][k];
#pragma unroll
      for (int n = 0; n < kHp / 16; ++n)
        if (16 * n + c < H) P[H * I + H + hr * H + 16 * n + c] = g2[n][k];
    }
    // the four row groups of a column
    gb1 += __shfl_xor(gb1, 16); gb1 += __shfl_xor(gb1, 32);
    gb2 += __shfl_xor(gb2, 16); gb2 += __shfl_xor(gb2, 32);
    gw3 += __shfl_xor(gw3, 16); gw3 += __shfl_xor(gw3, 32);
    if (q == 0 && on) {
      P[H * I + h] = gb1;
      P[H * I + H + H * H + h] = gb2;
      P[H * I + 2 * H + H * H + h] = gw3;
    }
    if (wv == 0) {
      for (int m = 8; m > 0; m >>= 1) { gb3 += __shfl_xor(gb3, m); gl += __shfl_xor(gl, m); }
      if (lane == 0) { P[np - 1] = gb3; P[np] = gl; }
    }
  }
}

// where the packed copies of a fused network's weights go
struct Packs {
  int I, H, ip;                      // ip 0: no packed copies (layer-by-layer network)
  unsigned short *w1, *w2, *w2t;
};
// parameter i as BF16: into the flat working copy and the packed ones
__device__ __forceinline__ void store_bf16(long long i, float v, hip_bfloat16* pb, const Packs& K) {
  const hip_bfloat16 b = hip_bfloat16(v);
  pb[i] = b;
  if (!K.ip) return;
  const long long o2 = (long long)K.H * K.I + K.H;
  if (i < (long long)K.H * K.I) {
    K.w1[(i / K.I) * K.ip + i % K.I] = b.data;
  } else if (i >= o2 && i < o2 + (long long)K.H * K.H) {
    const int m = (int)(i - o2), r = m / K.H, k = m % K.H;
    K.w2[r * kHp + k] = b.data;
    K.w2t[k * kHp + r] = b.data;
  }
}

// Adam on one FP32 master parameter, then the BF16 working copies
struct Adam {
  float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ void adam_step(long long i, float gi, float* p, float* m, float* v, const Adam& A,
                                          hip_bfloat16* pb, const Packs& K) {
  const float mi = A.b1 * m[i] + (1.f - A.b1) * gi;
  const float vi = A.b2 * v[i] + (1.f - A.b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - A.lr * (mi / A.c1) / (sqrtf(vi / A.c2) + A.eps);
  p[i] = pi;
  store_bf16(i, pi, pb, K);
}

// gradient and loss from the nb partial sums of k_mlp, added in a fixed order
// (4 strided groups, then the groups), and with STEP the Adam update.  The
// partials are read once, 256 B per wave and part.
template <bool STEP>
__global__ void __launch_bounds__(256) k_mlp_reduce(int np, int nb, const float* __restrict__ part, float* g,
                                                    float* loss, float* p, float* m, float* v, Adam A,
                                                    hip_bfloat16* pb, Packs K) {
  __shared__ float s_sum[4][64];
  const int c = threadIdx.x & 63, r = threadIdx.x >> 6, i = blockIdx.x * 64 + c;
  float s = 0.f;
  if (i <= np)
#pragma unroll 4
    for (int b = r; b < nb; b += 4) s += part[(size_t)b * (np + 1) + i];
  s_sum[r][c] = s;
  __syncthreads();
  if (r != 0 || i > np) return;
  const float t = (s_sum[0][c] + s_sum[1][c]) + (s_sum[2][c] + s_sum[3][c]);
  if (i == np) { *loss = t; return; }
  if (STEP) adam_step(i, t, p, m, v, A, pb, K);
  else g[i] = t;
}

// Adam on all parameters from the gradient array (layer-by-layer networks)
__global__ void k_adam(long long n, float* p, const float* g, float* m, float* v, Adam A, hip_bfloat16* pb, Packs K) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) adam_step(i, g[i], p, m, v, A, pb, K);
}

__global__ void k_to_bf16(long long n, const float* p, hip_bfloat16* pb, Packs K) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) store_bf16(i, p[i], pb, K);
}

// rows idx[0..B) of X (n_in) and T into the batch buffers
__global__ void k_gather(int B, int n_in, const int* idx, const float* X, const float* T, float* xb, float* tb) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= B * n_in) return;
  const int b = i / n_in, c = i % n_in;
  xb[i] = X[(size_t)idx[b] * n_in + c];
  if (c == 0) tb[b] = T[idx[b]];
}

inline int nblk(long long n, int t) { return (int)((n + t - 1) / t); }

}  // namespace

struct qmi_mlp {
  int device = 0;
  int n_in = 0, H = 0;
  hipStream_t s = nullptr;
  // parameters, in the order W1 (H x n_in), b1 (H), W2 (H x H), b2 (H), W3 (1 x H), b3 (1)
  long long np = 0;
  long long o_w1 = 0, o_b1 = 0, o_w2 = 0, o_b2 = 0, o_w3 = 0, o_b3 = 0;
  float* p = nullptr;           // FP32 master
  hip_bfloat16* pb = nullptr;   // BF16 working copy
  float *g = nullptr, *m = nullptr, *v = nullptr;
  Packs pk{};                   // packed weights of a fused network (pk.ip != 0)
  float* part = nullptr;        // fused: partial gradients of kPartBlocks blocks, from the first gradient on
  long long step = 0;
  // activations for a batch of up to cap rows
  int cap = 0;
  float *x = nullptr, *t = nullptr, *z1 = nullptr, *a1 = nullptr, *z2 = nullptr, *a2 = nullptr, *z3 = nullptr,
        *y = nullptr, *dz3 = nullptr, *da2 = nullptr, *dz2 = nullptr, *da1 = nullptr, *dz1 = nullptr,
        *lossv = nullptr, *loss = nullptr;
  // training set and row order of qmi_mlp_train, kept between calls and
  // replaced by larger ones
  long long tcap = 0;
  void* tbuf = nullptr;
  std::vector<void*> bufs;
  ~qmi_mlp() {
    if (tbuf) (void)hipFree(tbuf);
    for (void* b : bufs) (void)hipFree(b);
    if (s) (void)hipStreamDestroy(s);
  }
  template <typename T>
  int alloc(T** out, size_t n) {
    void* ptr = nullptr;
    if (hipMalloc(&ptr, std::max<size_t>(1, n) * sizeof(T)) != hipSuccess) return mlp_err(-101, "out of device memory");
    bufs.push_back(ptr);
    *out = (T*)ptr;
    return 0;
  }
};

namespace {

int ensure_batch(qmi_mlp* M, int B) {
  if (B <= M->cap) return 0;
  const int H = M->H;
  int rc;
  float** f[] = {&M->z1, &M->a1, &M->z2, &M->a2, &M->dz2, &M->da2, &M->da1, &M->dz1};
  for (float** q : f)
    if (!M->pk.ip && (rc = M->alloc(q, (size_t)B * H)) != 0) return rc;   // a fused network keeps no activations
  if ((rc = M->alloc(&M->x, (size_t)B * M->n_in)) != 0) return rc;
  for (float** q : {&M->t, &M->z3, &M->y, &M->dz3, &M->lossv})
    if ((rc = M->alloc(q, (size_t)B)) != 0) return rc;
  if ((rc = M->alloc(&M->loss, 1)) != 0) return rc;
  M->cap = B;
  return 0;
}

// the buffer of a fused network's partial gradients (21 MB for 34 inputs and 128
// hidden units), which a network that only predicts has no use for
int ensure_part(qmi_mlp* M) {
  if (!M->pk.ip || M->part) return 0;
  return M->alloc(&M->part, (size_t)kPartBlocks * (M->np + 1));
}

template <typename TA_, typename TB_, bool TA, bool TB>
void gemm(hipStream_t s, int Mr, int N, int K, float alpha, const TA_* A, int lda, const TB_* B, int ldb, float beta,
          float* C, int ldc) {
  dim3 grid(nblk(N, 16), nblk(Mr, 16));
  k_gemm<TA_, TB_, TA, TB><<<grid, 256, 0, s>>>(Mr, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
}

// activations of one forward pass: B x H (z1, a1, z2, a2) and B (z3)
struct Act {
  float *z1, *a1, *z2, *a2, *z3;
};

Net net_of(const qmi_mlp* M) {
  return Net{M->n_in, M->H, M->pk.w1, M->pk.w2, M->pk.w2t, M->pb + M->o_w3, M->p + M->o_b1, M->p + M->o_b2, M->p + M->o_b3};
}

// fused forward pass: one launch, no activations in memory
void fused_forward(qmi_mlp* M, hipStream_t s, int B, const float* x, float* y) {
  const int nb = nblk(B, kTileRows);
  if (M->pk.ip == 64) k_mlp<64, false><<<nb, kFusedBlock, 0, s>>>(B, net_of(M), x, nullptr, nullptr, y, nullptr);
  else k_mlp<128, false><<<nb, kFusedBlock, 0, s>>>(B, net_of(M), x, nullptr, nullptr, y, nullptr);
}
// fused gradient pass over rows idx[0..B) (all rows without idx) of X and T
// into M->part; returns the number of partial sums.  More blocks than
// kPartBlocks (one per CU) would only lengthen the reduction.
int fused_gradient(qmi_mlp* M, int B, const float* X, const float* T, const int* idx) {
  const int nb = std::min(nblk(B, kTileRows), kPartBlocks);
  if (M->pk.ip == 64) k_mlp<64, true><<<nb, kFusedBlock, 0, M->s>>>(B, net_of(M), X, T, idx, nullptr, M->part);
  else k_mlp<128, true><<<nb, kFusedBlock, 0, M->s>>>(B, net_of(M), X, T, idx, nullptr, M->part);
  return nb;
}

// forward pass of B rows x[B x n_in] into y[B] on stream s, activations in
// `a`; with targets t also the loss terms and dz3
void forward_on(qmi_mlp* M, hipStream_t s, int B, const float* x, const Act& a, float* y, const float* t,
                float* dz3, float* lossv) {
  const int H = M->H, I = M->n_in;
  const hip_bfloat16* W1 = M->pb + M->o_w1;
  const hip_bfloat16* W2 = M->pb + M->o_w2;
  const hip_bfloat16* W3 = M->pb + M->o_w3;
  gemm<float, hip_bfloat16, false, true>(s, B, H, I, 1.f, x, I, W1, I, 0.f, a.z1, H);   // x W1^T
  k_bias_silu<<<nblk((long long)B * H, 256), 256, 0, s>>>(B, H, a.z1, M->p + M->o_b1, a.a1);
  gemm<float, hip_bfloat16, false, true>(s, B, H, H, 1.f, a.a1, H, W2, H, 0.f, a.z2, H);  // a1 W2^T
  k_bias_silu<<<nblk((long long)B * H, 256), 256, 0, s>>>(B, H, a.z2, M->p + M->o_b2, a.a2);
  gemm<float, hip_bfloat16, false, true>(s, B, 1, H, 1.f, a.a2, H, W3, H, 0.f, a.z3, 1);  // a2 W3^T
  k_out<<<nblk(B, 256), 256, 0, s>>>(B, a.z3, M->p + M->o_b3, y, t, dz3, lossv);
}

// forward pass of B rows in M->x; with targets (M->t) also the loss and dz3
void forward(qmi_mlp* M, int B, bool with_t) {
  if (M->pk.ip && !with_t) {
    fused_forward(M, M->s, B, M->x, M->y);
    return;
  }
  forward_on(M, M->s, B, M->x, Act{M->z1, M->a1, M->z2, M->a2, M->z3}, M->y, with_t ? M->t : nullptr, M->dz3,
             M->lossv);
}

// Scratch of qmi_mlp_forward_noalloc: the activations of one forward pass,
// B x (4H + 1) floats, in a fixed device array (4 MiB on every device the
// library runs on, held until the process ends).  Host code never passes the
// array's name to a kernel: it uses the address hipGetSymbolAddress returns
// for the current device, kept per device in scratch_ptr.
constexpr long long kScratchFloats = 1LL << 20;
__device__ __align__(256) float scratch[kScratchFloats];
constexpr int kMaxDevices = 64;
float* scratch_ptr[kMaxDevices] = {};

// set up scratch_ptr for `device`, which must be current
int scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices) return mlp_err(-1, "device number beyond the scratch table");
  if (scratch_ptr[device]) return 0;
  void* ptr = nullptr;
  MLP_OK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  if (!ptr) return mlp_err(-100, "no address for the scratch array");
  scratch_ptr[device] = (float*)ptr;
  return 0;
}

// gradient of the mean squared error into M->g (after forward with targets)
void backward(qmi_mlp* M, int B) {
  const int H = M->H, I = M->n_in;
  hipStream_t s = M->s;
  const hip_bfloat16* W2 = M->pb + M->o_w2;
  const hip_bfloat16* W3 = M->pb + M->o_w3;
  float* g = M->g;
  // output layer
  gemm<float, float, true, false>(s, 1, H, B, 1.f, M->dz3, 1, M->a2, H, 0.f, g + M->o_w3, H);  // dz3^T a2
  k_sum<<<1, 256, 0, s>>>(B, M->dz3, g + M->o_b3);
  gemm<float, hip_bfloat16, false, false>(s, B, H, 1, 1.f, M->dz3, 1, W3, H, 0.f, M->da2, H);  // dz3 W3
  k_silu_back<<<nblk((long long)B * H, 256), 256, 0, s>>>(B * H, M->z2, M->da2, M->dz2);
  // hidden layer 2
  gemm<float, float, true, false>(s, H, H, B, 1.f, M->dz2, H, M->a1, H, 0.f, g + M->o_w2, H);  // dz2^T a1
  k_colsum<<<nblk(H, 64), 64 * kSumGroups, 0, s>>>(B, H, M->dz2, g + M->o_b2);
  gemm<float, hip_bfloat16, false, false>(s, B, H, H, 1.f, M->dz2, H, W2, H, 0.f, M->da1, H);  // dz2 W2
  k_silu_back<<<nblk((long long)B * H, 256), 256, 0, s>>>(B * H, M->z1, M->da1, M->dz1);
  // hidden layer 1
  gemm<float, float, true, false>(s, H, I, B, 1.f, M->dz1, H, M->x, I, 0.f, g + M->o_w1, I);  // dz1^T x
  k_colsum<<<nblk(H, 64), 64 * kSumGroups, 0, s>>>(B, H, M->dz1, g + M->o_b1);
}

}  // namespace

extern "C" {

const char* qmi_mlp_last_error(void) { return g_mlp_err.c_str(); }

int qmi_mlp_create(int hip_device, int n_in, int n_hidden, unsigned long long seed, qmi_mlp** out) {
  if (!out || n_in < 1 || n_in > 4096 || n_hidden < 1 || n_hidden > 4096) return mlp_err(-1, "invalid MLP shape");
  int ndev = 0;
  MLP_OK(hipGetDeviceCount(&ndev));
  if (hip_device < 0 || hip_device >= ndev) return mlp_err(-1, "invalid HIP device");
  MLP_OK(hipSetDevice(hip_device));
  auto* M = new qmi_mlp();
  M->device = hip_device;
  M->n_in = n_in;
  M->H = n_hidden;
  const long long H = n_hidden, I = n_in;
  M->o_w1 = 0;
  M->o_b1 = H * I;
  M->o_w2 = M->o_b1 + H;
  M->o_b2 = M->o_w2 + H * H;
  M->o_w3 = M->o_b2 + H;
  M->o_b3 = M->o_w3 + H;
  M->np = M->o_b3 + 1;
  int rc;
  if (hipStreamCreate(&M->s) != hipSuccess) { delete M; return mlp_err(-100, "stream"); }
  if ((rc = M->alloc(&M->p, M->np)) || (rc = M->alloc(&M->pb, M->np)) || (rc = M->alloc(&M->g, M->np)) ||
      (rc = M->alloc(&M->m, M->np)) || (rc = M->alloc(&M->v, M->np))) {
    delete M;
    return rc;
  }
  // fused up to 128 inputs and hidden units: the weight gradients then stay
  // in 64 accumulator registers a lane and the rows in 25 KB of LDS.  At
  // these sizes the layer-by-layer form takes 2 to 36 times as long (see
  // k_mlp); beyond them the accumulators no longer fit
  if (n_hidden <= kHp && n_in <= 128) {
    M->pk = Packs{n_in, n_hidden, n_in <= 64 ? 64 : 128, nullptr, nullptr, nullptr};
    unsigned short* w = nullptr;
    const size_t n1 = (size_t)kHp * M->pk.ip, n2 = (size_t)kHp * kHp;
    if ((rc = M->alloc(&w, n1 + 2 * n2)) != 0) {
      delete M;
      return rc;
    }
    M->pk.w1 = w;
    M->pk.w2 = w + n1;
    M->pk.w2t = w + n1 + n2;
    if (hipMemset(w, 0, (n1 + 2 * n2) * 2) != hipSuccess) { delete M; return mlp_err(-100, "init"); }
  }
  // He-style uniform initialisation from the seed, biases zero
  std::vector<float> h(M->np, 0.f);
  std::mt19937_64 rng(seed);
  auto fill = [&](long long off, long long n, long long fan_in) {
    const float a = std::sqrt(6.0f / (float)fan_in);
    std::uniform_real_distribution<float> u(-a, a);
    for (long long k = 0; k < n; ++k) h[off + k] = u(rng);
  };
  fill(M->o_w1, H * I, I);
  fill(M->o_w2, H * H, H);
  fill(M->o_w3, H, H);
  std::vector<float> zero(M->np, 0.f);
  if (hipMemcpy(M->p, h.data(), M->np * 4, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(M->m, zero.data(), M->np * 4, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(M->v, zero.data(), M->np * 4, hipMemcpyHostToDevice) != hipSuccess) {
    delete M;
    return mlp_err(-100, "upload");
  }
  k_to_bf16<<<nblk(M->np, 256), 256, 0, M->s>>>(M->np, M->p, M->pb, M->pk);
  if (hipStreamSynchronize(M->s) != hipSuccess) { delete M; return mlp_err(-100, "init"); }
  {
    // the fixed scratch array of qmi_mlp_forward_noalloc on this device
    static std::mutex mu;
    std::lock_guard<std::mutex> lock(mu);
    if ((rc = scratch_init(hip_device)) != 0) { delete M; return rc; }
  }
  *out = M;
  return 0;
}

long long qmi_mlp_num_params(qmi_mlp* M) { return M ? M->np : -1; }

int qmi_mlp_get_params(qmi_mlp* M, float* params, long long cap) {
  if (!M || !params) return mlp_err(-1, "null argument");
  if (cap < M->np) return mlp_err(-3, "buffer too small");
  MLP_OK(hipSetDevice(M->device));
  MLP_OK(hipMemcpy(params, M->p, M->np * 4, hipMemcpyDeviceToHost));
  return 0;
}

int qmi_mlp_set_params(qmi_mlp* M, const float* params, long long n) {
  if (!M || !params) return mlp_err(-1, "null argument");
  if (n != M->np) return mlp_err(-3, "wrong number of parameters");
  MLP_OK(hipSetDevice(M->device));
  MLP_OK(hipMemcpy(M->p, params, n * 4, hipMemcpyHostToDevice));
  k_to_bf16<<<nblk(M->np, 256), 256, 0, M->s>>>(M->np, M->p, M->pb, M->pk);
  MLP_OK(hipStreamSynchronize(M->s));
  return 0;
}

int qmi_mlp_forward(qmi_mlp* M, const float* x, int batch, float* y) {
  if (!M || !x || !y || batch < 1) return mlp_err(-1, "invalid argument");
  MLP_OK(hipSetDevice(M->device));
  int rc;
  if ((rc = ensure_batch(M, batch)) != 0) return rc;
  MLP_OK(hipMemcpyAsync(M->x, x, (size_t)batch * M->n_in * 4, hipMemcpyHostToDevice, M->s));
  forward(M, batch, false);
  MLP_OK(hipGetLastError());
  MLP_OK(hipMemcpyAsync(y, M->y, (size_t)batch * 4, hipMemcpyDeviceToHost, M->s));
  MLP_OK(hipStreamSynchronize(M->s));
  return 0;
}

int qmi_mlp_forward_noalloc(qmi_mlp* M, const float* d_x, int batch, float* d_y, void* stream) {
  if (!M || !d_x || !d_y || batch < 1) return mlp_err(-1, "invalid argument");
  const long long per_row = 4LL * M->H + 1;
  if ((long long)batch * per_row > kScratchFloats)
    return mlp_err(-3, "batch of " + std::to_string(batch) + " rows exceeds the scratch of " +
                           std::to_string(kScratchFloats / per_row) + " rows for this network");
  float* base = M->device >= 0 && M->device < kMaxDevices ? scratch_ptr[M->device] : nullptr;
  if (!base) return mlp_err(-2, "scratch not set up for this device");
  MLP_OK(hipSetDevice(M->device));
  const long long BH = (long long)batch * M->H;
  const Act a{base, base + BH, base + 2 * BH, base + 3 * BH, base + 4 * BH};
  const hipStream_t s = stream ? (hipStream_t)stream : M->s;
  if (M->pk.ip) fused_forward(M, s, batch, d_x, d_y);
  else forward_on(M, s, batch, d_x, a, d_y, nullptr, nullptr, nullptr);
  MLP_OK(hipGetLastError());
  return 0;
}

int qmi_mlp_grad(qmi_mlp* M, const float* x, const float* t, int batch, float* loss, float* grad) {
  if (!M || !x || !t || batch < 1) return mlp_err(-1, "invalid argument");
  MLP_OK(hipSetDevice(M->device));
  int rc;
  if ((rc = ensure_batch(M, batch)) != 0 || (rc = ensure_part(M)) != 0) return rc;
  MLP_OK(hipMemcpyAsync(M->x, x, (size_t)batch * M->n_in * 4, hipMemcpyHostToDevice, M->s));
  MLP_OK(hipMemcpyAsync(M->t, t, (size_t)batch * 4, hipMemcpyHostToDevice, M->s));
  if (M->pk.ip) {
    const int nb = fused_gradient(M, batch, M->x, M->t, nullptr);
    k_mlp_reduce<false><<<nblk(M->np + 1, 64), 256, 0, M->s>>>((int)M->np, nb, M->part, M->g, M->loss, M->p, M->m, M->v,
                                                               Adam{}, M->pb, M->pk);
  } else {
    forward(M, batch, true);
    backward(M, batch);
    k_sum<<<1, 256, 0, M->s>>>(batch, M->lossv, M->loss);
  }
  MLP_OK(hipGetLastError());
  float l = 0.f;
  MLP_OK(hipMemcpyAsync(&l, M->loss, 4, hipMemcpyDeviceToHost, M->s));
  if (grad) MLP_OK(hipMemcpyAsync(grad, M->g, M->np * 4, hipMemcpyDeviceToHost, M->s));
  MLP_OK(hipStreamSynchronize(M->s));
  if (loss) *loss = l / (float)batch;
  return 0;
}

int qmi_mlp_train(qmi_mlp* M, const float* X, const float* T, int n, int epochs, int batch, float lr,
                  unsigned long long seed, float* final_loss) {
  if (!M || !X || !T || n < 1 || epochs < 0 || batch < 1) return mlp_err(-1, "invalid argument");
  MLP_OK(hipSetDevice(M->device));
  batch = std::min(batch, n);
  int rc;
  if ((rc = ensure_batch(M, batch)) != 0 || (rc = ensure_part(M)) != 0) return rc;
  // the training set, the row order and the last pass's losses stay on the
  // device for the whole call
  const size_t nx = (size_t)n * M->n_in, per_pass = (size_t)(n / batch);
  const size_t need = (nx + 2 * (size_t)n + per_pass) * 4;
  if ((long long)need > M->tcap) {
    if (M->tbuf) MLP_OK(hipFree(M->tbuf));
    M->tbuf = nullptr;
    M->tcap = 0;
    if (hipMalloc(&M->tbuf, need) != hipSuccess) return mlp_err(-101, "out of device memory");
    M->tcap = (long long)need;
  }
  float* dX = (float*)M->tbuf;
  float* dT = dX + nx;
  int* didx = (int*)(dT + n);
  float* dloss = (float*)(didx + n);
  MLP_OK(hipMemcpy(dX, X, nx * 4, hipMemcpyHostToDevice));
  MLP_OK(hipMemcpy(dT, T, (size_t)n * 4, hipMemcpyHostToDevice));
  std::vector<int> order(n);
  for (int k = 0; k < n; ++k) order[k] = k;
  std::mt19937_64 rng(seed);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int ep = 0; ep < epochs; ++ep) {
    std::shuffle(order.begin(), order.end(), rng);
    MLP_OK(hipMemcpyAsync(didx, order.data(), (size_t)n * 4, hipMemcpyHostToDevice, M->s));
    for (int b0 = 0, kb = 0; b0 + batch <= n; b0 += batch, ++kb) {
      ++M->step;
      const Adam A{lr, b1, b2, eps, 1.f - std::pow(b1, (float)M->step), 1.f - std::pow(b2, (float)M->step)};
      if (M->pk.ip) {
        const int nb = fused_gradient(M, batch, dX, dT, didx + b0);
        k_mlp_reduce<true><<<nblk(M->np + 1, 64), 256, 0, M->s>>>((int)M->np, nb, M->part, M->g, dloss + kb, M->p, M->m,
                                                                  M->v, A, M->pb, M->pk);
        continue;
      }
      k_gather<<<nblk((long long)batch * M->n_in, 256), 256, 0, M->s>>>(batch, M->n_in, didx + b0, dX, dT, M->x, M->t);
      forward(M, batch, true);
      backward(M, batch);
      k_adam<<<nblk(M->np, 256), 256, 0, M->s>>>(M->np, M->p, M->g, M->m, M->v, A, M->pb, M->pk);
      if (ep == epochs - 1) k_sum<<<1, 256, 0, M->s>>>(batch, M->lossv, dloss + kb);
    }
    MLP_OK(hipGetLastError());
  }
  double last = 0.0;
  if (epochs > 0) {
    std::vector<float> l(per_pass);
    MLP_OK(hipMemcpyAsync(l.data(), dloss, per_pass * 4, hipMemcpyDeviceToHost, M->s));
    MLP_OK(hipStreamSynchronize(M->s));
    for (float v : l) last += v;
    last /= (double)((n / batch) * batch);
  }
  MLP_OK(hipStreamSynchronize(M->s));
  if (final_loss) *final_loss = (float)last;
  return 0;
}

void qmi_mlp_destroy(qmi_mlp* M) { delete M; }

}  // extern "C"
