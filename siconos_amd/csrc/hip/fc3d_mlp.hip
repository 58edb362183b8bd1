// fc3d_mlp.hip — the learned warm start's network (no reference counterpart).
//
// MLP 22 -> 128 -> 128 -> 128 -> 3 with GELU.  Every product runs on the
// matrix cores as v_mfma_f32_16x16x16bf16_1k (BF16 operands, FP32
// accumulation):
//   forward         four wavefronts carry 16 contacts through all layers, a
//                   quarter of each layer's outputs a wave, activations in
//                   LDS (16 x 128 BF16 per buffer);
//   backward        goes on in the same workgroup from the pre-activations in
//                   its registers, dA = dZ W with W^T kept in HBM as BF16;
//   gradients       one launch: a wavefront per 16 x 16 tile of a dW, the
//                   minibatch as the MFMA reduction (activations and dZ are
//                   stored feature-major so that both operands are
//                   contiguous), and a wavefront per bias;
//   step            one launch: Adam on the FP32 master weights and the BF16
//                   re-cast of W and W^T.
// A minibatch of 1024 rows is 64 workgroups: the chip is mostly idle and a
// step is the sum of its kernels' chains, so there are three of them.  As
// sixteen launches (the rows' gather, a wave per 16 contacts, Z through HBM, a
// launch per matrix) a step took 210 us; it takes ~50.
//
// MFMA 16x16x16 operand layout (wave64, lane l, i = 0..3):
//   A (M x K):  lane holds A[l % 16][4 (l / 16) + i]
//   B (K x N):  lane holds B[4 (l / 16) + i][l % 16]
//   D (M x N):  lane holds D[4 (l / 16) + i][l % 16]
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "fc3d_internal.hpp"
#include "fc3d_mlp.hpp"

namespace fc3d {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16;

// FP32 -> BF16, round to nearest even (finite inputs)
__host__ __device__ __forceinline__ bf16 f2bf(float f) {
  unsigned u = __builtin_bit_cast(unsigned, f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__host__ __device__ __forceinline__ float bf2f(bf16 b) {
  return __builtin_bit_cast(float, (unsigned)b << 16);
}

__device__ __forceinline__ float gelu(float z) {
  return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));
}
__device__ __forceinline__ float gelu_grad(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) +
         z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// parameter offsets in the FP32 master vector
constexpr int OW1 = 0, OB1 = OW1 + MLP_H * MLP_K1, OW2 = OB1 + MLP_H, OB2 = OW2 + MLP_H * MLP_H,
              OW3 = OB2 + MLP_H, OB3 = OW3 + MLP_H * MLP_H, OW4 = OB3 + MLP_H,
              OB4 = OW4 + MLP_NOP * MLP_H, NPARAM = OB4 + MLP_NOP;
static_assert(NPARAM == MLP_NPARAMS, "parameter count");

struct MlpWeights {
  const bf16* w[4];   // [n][k]
  const bf16* wt[4];  // [k][n]
  const float* b[4];
};

// acc[t] = act x W^T for the 16 x 16 output tiles t0 .. t0 + NT - 1, where act
// is [16][K] (LDS) and W is [rows = outputs][K].
template <int K, int NT>
__device__ __forceinline__ void wave_dense(const bf16* act, const bf16* __restrict__ W, int t0,
                                           f32x4* acc) {
  const int l = threadIdx.x & 63, row = l & 15, kq = l >> 4;
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += 16) {
    const bf16x4 a = *reinterpret_cast<const bf16x4*>(&act[row * K + k0 + 4 * kq]);
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const bf16x4 b =
          *reinterpret_cast<const bf16x4*>(&W[(size_t)((t0 + t) * 16 + row) * K + k0 + 4 * kq]);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t], 0, 0, 0);
    }
  }
}

struct TrainBufs {
  int bsz;              // rows of the pass (multiple of 64)
  bf16* At[4];          // feature-major layer inputs: At[0] [32][bsz], At[l] [128][bsz]
  bf16* dZt[4];         // feature-major dZ: [128][bsz] for l = 0..2, [16][bsz] for l = 3
  const int* idx;       // row r of the pass is row idx[r] of X and target; null: row r
  const float* target;  // [rows][3]
  float* loss_part;     // per 16 rows: sum of squared errors
};

// Four consecutive rows of one feature, feature-major (8-byte aligned: the
// pass has a multiple of 64 rows).
__device__ __forceinline__ void store4(bf16* p, const bf16* v) {
  *reinterpret_cast<bf16x4*>(p) = bf16x4{(short)v[0], (short)v[1], (short)v[2], (short)v[3]};
}

// A hidden layer of the workgroup's 16 rows: this wave's two output tiles from
// `in`, activations to `out`, pre-activations to z.
template <int K>
__device__ __forceinline__ void hidden_layer(const bf16* in, const bf16* __restrict__ W,
                                             const float* __restrict__ b, int wave, bf16* out,
                                             f32x4* z, bf16* At, int bsz, int m0) {
  const int l = threadIdx.x & 63, col = l & 15, rq = l >> 4;
  f32x4 acc[2];
  wave_dense<K, 2>(in, W, 2 * wave, acc);
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int nn = (2 * wave + t) * 16 + col;
    bf16 a[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      z[t][i] = acc[t][i] + b[nn];
      a[i] = f2bf(gelu(z[t][i]));
      out[(4 * rq + i) * MLP_H + nn] = a[i];
    }
    if (At) store4(&At[(size_t)nn * bsz + m0 + 4 * rq], a);
  }
}

// Forward pass, 16 contacts per workgroup of 4 waves; X is [>= 16 blocks][32]
// standardised BF16 inputs, y [n][3].
__global__ __launch_bounds__(256) void k_mlp_forward(int n, const bf16* __restrict__ X,
                                                     MlpWeights w, float* __restrict__ y) {
  __shared__ __attribute__((aligned(16))) bf16 a0[16 * MLP_H], a1[16 * MLP_H];
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int m0 = blockIdx.x * 16;
  for (int e = threadIdx.x; e < 16 * MLP_K1; e += 256) a0[e] = X[(size_t)m0 * MLP_K1 + e];
  __syncthreads();
  f32x4 z[2];
  hidden_layer<MLP_K1>(a0, w.w[0], w.b[0], wave, a1, z, nullptr, 0, 0);
  __syncthreads();
  hidden_layer<MLP_H>(a1, w.w[1], w.b[1], wave, a0, z, nullptr, 0, 0);
  __syncthreads();
  hidden_layer<MLP_H>(a0, w.w[2], w.b[2], wave, a1, z, nullptr, 0, 0);
  __syncthreads();
  if (wave) return;
  f32x4 acc[1];
  wave_dense<MLP_H, 1>(a1, w.w[3], 0, acc);
  const int col = l & 15, rq = l >> 4;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int m = 4 * rq + i;
    const float v = acc[0][i] + w.b[3][col];
    if (m0 + m < n && col < MLP_NO) y[(size_t)(m0 + m) * MLP_NO + col] = v;
  }
}

// Forward and backward of the data path for the mean squared error over the
// first `nvalid` rows, 16 rows per workgroup: dZ of the output layer, then dA =
// dZ W and dZ = dA gelu'(Z) down to the first layer.  Layer inputs and dZ go
// out feature-major in BF16.
__global__ __launch_bounds__(256) void k_mlp_fwd_bwd(int nvalid, const bf16* __restrict__ X,
                                                     MlpWeights w, TrainBufs tb) {
  __shared__ __attribute__((aligned(16))) bf16 a0[16 * MLP_H], a1[16 * MLP_H], d3[16 * MLP_NOP];
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, col = l & 15, rq = l >> 4;
  const int m0 = blockIdx.x * 16;
  for (int e = threadIdx.x; e < 16 * MLP_K1; e += 256) {
    const int m = e / MLP_K1, k = e % MLP_K1;
    const int src = tb.idx ? tb.idx[m0 + m] : m0 + m;
    const bf16 x = X[(size_t)src * MLP_K1 + k];
    a0[e] = x;
    tb.At[0][(size_t)k * tb.bsz + m0 + m] = x;
  }
  __syncthreads();
  f32x4 z0[2], z1[2], z2[2], acc[2];
  hidden_layer<MLP_K1>(a0, w.w[0], w.b[0], wave, a1, z0, tb.At[1], tb.bsz, m0);
  __syncthreads();
  hidden_layer<MLP_H>(a1, w.w[1], w.b[1], wave, a0, z1, tb.At[2], tb.bsz, m0);
  __syncthreads();
  hidden_layer<MLP_H>(a0, w.w[2], w.b[2], wave, a1, z2, tb.At[3], tb.bsz, m0);
  __syncthreads();
  if (wave == 0) {
    wave_dense<MLP_H, 1>(a1, w.w[3], 0, acc);
    const float scale = 2.0f / (float)(nvalid * MLP_NO);
    float lsum = 0.f;
    bf16 gb[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int m = 4 * rq + i;
      const float v = acc[0][i] + w.b[3][col];
      float g = 0.f;
      if (col < MLP_NO && m0 + m < nvalid) {
        const int src = tb.idx ? tb.idx[m0 + m] : m0 + m;
        const float diff = v - tb.target[(size_t)src * MLP_NO + col];
        g = scale * diff;
        lsum += diff * diff;
      }
      gb[i] = f2bf(g);
      d3[m * MLP_NOP + col] = gb[i];
    }
    store4(&tb.dZt[3][(size_t)col * tb.bsz + m0 + 4 * rq], gb);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, 64);
    if (l == 0) tb.loss_part[blockIdx.x] = lsum;
  }
  __syncthreads();
  // dZ of a layer from dA (acc) and its pre-activations
  auto dz = [&](const f32x4* z, bf16* out, bf16* dZt) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int nn = (2 * wave + t) * 16 + col;
      bf16 g[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        g[i] = f2bf(acc[t][i] * gelu_grad(z[t][i]));
        if (out) out[(4 * rq + i) * MLP_H + nn] = g[i];
      }
      store4(&dZt[(size_t)nn * tb.bsz + m0 + 4 * rq], g);
    }
  };
  // dA of the third hidden layer = dZ4 W4 (reduction over the 16 outputs)
  wave_dense<MLP_NOP, 2>(d3, w.wt[3], 2 * wave, acc);
  dz(z2, a0, tb.dZt[2]);
  __syncthreads();
  wave_dense<MLP_H, 2>(a0, w.wt[2], 2 * wave, acc);
  dz(z1, a1, tb.dZt[1]);
  __syncthreads();
  wave_dense<MLP_H, 2>(a1, w.wt[1], 2 * wave, acc);
  dz(z0, nullptr, tb.dZt[0]);
}

// All gradients: dW[n][k] = sum_m dZ[m][n] A[m][k], one 16 x 16 tile per wave
// (the loads of eight steps in flight), then db[n] = sum_m dZ[m][n], one wave
// per output with fixed-order lane sums.
constexpr int MLP_TILES[4] = {(MLP_H / 16) * (MLP_K1 / 16), (MLP_H / 16) * (MLP_H / 16),
                              (MLP_H / 16) * (MLP_H / 16), (MLP_NOP / 16) * (MLP_H / 16)};
constexpr int MLP_ALL_TILES = MLP_TILES[0] + MLP_TILES[1] + MLP_TILES[2] + MLP_TILES[3];
constexpr int MLP_GRAD_WAVES = MLP_ALL_TILES + 3 * MLP_H + MLP_NOP;
__global__ __launch_bounds__(256) void k_mlp_grads(TrainBufs tb, float* __restrict__ grads) {
  const int l = threadIdx.x & 63, bsz = tb.bsz;
  int wv = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (wv >= MLP_GRAD_WAVES) return;
  constexpr int woff[4] = {OW1, OW2, OW3, OW4}, boff[4] = {OB1, OB2, OB3, OB4};
  if (wv < MLP_ALL_TILES) {
    int layer = 0;
    while (wv >= MLP_TILES[layer]) wv -= MLP_TILES[layer++];
    const int kin = layer == 0 ? MLP_K1 : MLP_H, ktiles = kin / 16;
    const int n0 = (wv / ktiles) * 16, k0 = (wv % ktiles) * 16;
    const int r = l & 15, q = l >> 4;
    const bf16* __restrict__ pa = tb.dZt[layer] + (size_t)(n0 + r) * bsz + 4 * q;
    const bf16* __restrict__ pb = tb.At[layer] + (size_t)(k0 + r) * bsz + 4 * q;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int m0 = 0; m0 < bsz; m0 += 16) {
      const bf16x4 a = *reinterpret_cast<const bf16x4*>(pa + m0);
      const bf16x4 b = *reinterpret_cast<const bf16x4*>(pb + m0);
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    float* dW = grads + woff[layer];
#pragma unroll
    for (int i = 0; i < 4; i++) dW[(size_t)(n0 + 4 * q + i) * kin + k0 + r] = acc[i];
    return;
  }
  wv -= MLP_ALL_TILES;
  const int layer = wv / MLP_H, nn = wv % MLP_H;  // (the last layer has 16 outputs)
  const bf16* __restrict__ d = tb.dZt[layer] + (size_t)nn * bsz;
  float s = 0.f;
#pragma unroll 8
  for (int m = l; m < bsz; m += 64) s += bf2f(d[m]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (l == 0) grads[boff[layer] + nn] = s;
}

// Adam, and the BF16 copies of the weight it moved ([n][k] and [k][n]).
__global__ void k_adam(int np, float* __restrict__ p, const float* __restrict__ g,
                       float* __restrict__ m1, float* __restrict__ m2, float lr, float b1, float b2,
                       float c1, float c2, float eps, bf16* w0, bf16* wt0, bf16* w1, bf16* wt1,
                       bf16* w2, bf16* wt2, bf16* w3, bf16* wt3) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi;
  const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  const float v = p[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
  p[i] = v;
  auto cast = [&](int off, int nout, int kin, bf16* w, bf16* wt) {
    const int e = i - off;
    if (e < 0 || e >= nout * kin) return;
    const bf16 x = f2bf(v);
    w[e] = x;
    wt[(size_t)(e % kin) * nout + e / kin] = x;
  };
  cast(OW1, MLP_H, MLP_K1, w0, wt0);
  cast(OW2, MLP_H, MLP_H, w1, wt1);
  cast(OW3, MLP_H, MLP_H, w2, wt2);
  cast(OW4, MLP_NOP, MLP_H, w3, wt3);
}

// BF16 copies of one weight matrix, [n][k] and transposed [k][n]
__global__ void k_mlp_cast(const float* __restrict__ p, bf16* __restrict__ w, bf16* __restrict__ wt,
                           int nout, int kin) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nout * kin) return;
  const int nn = i / kin, k = i % kin;
  const bf16 v = f2bf(p[i]);
  w[i] = v;
  wt[(size_t)k * nout + nn] = v;
}

// X[npad][32] = bf16((f - mean) / std), zero for padded columns and rows >= n
__global__ void k_mlp_inputs(int n, int npad, const float* __restrict__ f,
                             const float* __restrict__ mean, const float* __restrict__ stdv,
                             bf16* __restrict__ X) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)npad * MLP_K1) return;
  const int m = (int)(i / MLP_K1), k = (int)(i % MLP_K1);
  X[i] = (k < MLP_NF && m < n) ? f2bf((f[(size_t)m * MLP_NF + k] - mean[k]) / stdv[k]) : (bf16)0;
}

}  // namespace fc3d

using namespace fc3d;

struct fc3d_hip_mlp {
  int device = 0;
  hipStream_t stream = nullptr;
  float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
  bf16* w[4] = {nullptr, nullptr, nullptr, nullptr};
  bf16* wt[4] = {nullptr, nullptr, nullptr, nullptr};
  float *mean = nullptr, *stdv = nullptr;
  long adam_t = 0;
  // training workspace for passes of up to ws_bsz rows
  int ws_bsz = 0;
  bf16* At[4] = {nullptr, nullptr, nullptr, nullptr};
  bf16* dZt[4] = {nullptr, nullptr, nullptr, nullptr};
  float* loss_part = nullptr;
};

namespace fc3d {

static const int kDims[4][2] = {{MLP_H, MLP_K1}, {MLP_H, MLP_H}, {MLP_H, MLP_H}, {MLP_NOP, MLP_H}};
static const int kWOff[4] = {OW1, OW2, OW3, OW4};
static const int kBOff[4] = {OB1, OB2, OB3, OB4};
static fc3d_hip_mlp* g_default_model = nullptr;

static MlpWeights mlp_weights(const fc3d_hip_mlp* m) {
  MlpWeights w;
  for (int k = 0; k < 4; k++) {
    w.w[k] = m->w[k];
    w.wt[k] = m->wt[k];
    w.b[k] = m->p + kBOff[k];
  }
  return w;
}

static int mlp_cast(fc3d_hip_mlp* m) {
  for (int k = 0; k < 4; k++) {
    const int n = kDims[k][0] * kDims[k][1];
    hipLaunchKernelGGL(k_mlp_cast, dim3((n + 255) / 256), dim3(256), 0, m->stream, m->p + kWOff[k],
                       m->w[k], m->wt[k], kDims[k][0], kDims[k][1]);
  }
  FC3D_HIP_TRY(hipGetLastError());
  return 0;
}

static void free_workspace(fc3d_hip_mlp* m) {
  for (int k = 0; k < 4; k++) {
    hipFree(m->At[k]);
    hipFree(m->dZt[k]);
    m->At[k] = m->dZt[k] = nullptr;
  }
  hipFree(m->loss_part);
  m->loss_part = nullptr;
  m->ws_bsz = 0;
}

static int mlp_workspace(fc3d_hip_mlp* m, int bsz) {
  if (m->ws_bsz >= bsz) return 0;
  FC3D_HIP_TRY(hipStreamSynchronize(m->stream));
  free_workspace(m);
  FC3D_HIP_TRY(hipMalloc(&m->At[0], sizeof(bf16) * bsz * MLP_K1));
  for (int k = 1; k < 4; k++) FC3D_HIP_TRY(hipMalloc(&m->At[k], sizeof(bf16) * bsz * MLP_H));
  for (int k = 0; k < 3; k++) FC3D_HIP_TRY(hipMalloc(&m->dZt[k], sizeof(bf16) * bsz * MLP_H));
  FC3D_HIP_TRY(hipMalloc(&m->dZt[3], sizeof(bf16) * bsz * MLP_NOP));
  FC3D_HIP_TRY(hipMalloc(&m->loss_part, sizeof(float) * (bsz / 16)));
  m->ws_bsz = bsz;
  return 0;
}

// Forward + backward over `bsz` rows (the first `nvalid` carry targets; idx
// picks them from X and T, null: the rows in order): gradients into m->g, loss
// partials into m->loss_part.
static int mlp_grad_pass(fc3d_hip_mlp* m, int nvalid, int bsz, const bf16* X, const float* T,
                         const int* idx) {
  TrainBufs tb;
  tb.bsz = bsz;
  for (int k = 0; k < 4; k++) {
    tb.At[k] = m->At[k];
    tb.dZt[k] = m->dZt[k];
  }
  tb.idx = idx;
  tb.target = T;
  tb.loss_part = m->loss_part;
  hipLaunchKernelGGL(k_mlp_fwd_bwd, dim3(bsz / 16), dim3(256), 0, m->stream, nvalid, X,
                     mlp_weights(m), tb);
  hipLaunchKernelGGL(k_mlp_grads, dim3((MLP_GRAD_WAVES + 3) / 4), dim3(256), 0, m->stream, tb,
                     m->g);
  FC3D_HIP_TRY(hipGetLastError());
  return 0;
}

static double sum_loss(fc3d_hip_mlp* m, int bsz, int* rc) {
  std::vector<float> lp((size_t)bsz / 16);
  hipError_t e = hipMemcpyAsync(lp.data(), m->loss_part, sizeof(float) * lp.size(),
                                hipMemcpyDeviceToHost, m->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
  if (e != hipSuccess) {
    set_error("fc3d_hip_mlp: loss read-back failed: %s", hipGetErrorString(e));
    *rc = NUMERICS_ERR_DEVICE;
    return 0.0;
  }
  double s = 0.0;
  for (float v : lp) s += v;
  return s;
}

int mlp_device(const fc3d_hip_mlp* m) { return m->device; }

int mlp_forward_device(fc3d_hip_mlp* m, int n, const float* feat, bf16* X, float* y,
                       hipStream_t s) {
  const int npad = (n + 63) / 64 * 64;
  hipLaunchKernelGGL(k_mlp_inputs, dim3((unsigned)(((size_t)npad * MLP_K1 + 255) / 256)),
                     dim3(256), 0, s, n, npad, feat, m->mean, m->stdv, X);
  hipLaunchKernelGGL(k_mlp_forward, dim3(npad / 16), dim3(256), 0, s, n, X, mlp_weights(m), y);
  FC3D_HIP_TRY(hipGetLastError());
  return 0;
}

// RAII list of device buffers freed on every return path
struct DevBufs {
  std::vector<void*> p;
  ~DevBufs() {
    for (void* q : p) hipFree(q);
  }
  template <typename T>
  hipError_t get(T** out, size_t n) {
    hipError_t e = hipMalloc(out, sizeof(T) * (n ? n : 1));
    if (e == hipSuccess) p.push_back(*out);
    return e;
  }
};

}  // namespace fc3d

extern "C" {

int fc3d_hip_mlp_create(uint64_t seed, int device, fc3d_hip_mlp** out) {
  if (!out) return NUMERICS_ERR_NULL_POINTER;
  *out = nullptr;
  int rc = use_device(device);
  if (rc) return rc;
  fc3d_hip_mlp* m = new fc3d_hip_mlp();
  m->device = device;
  auto fail = [&](int code) {
    fc3d_hip_mlp_destroy(m);
    return code;
  };
#define MLP_TRY(expr)                                                                      \
  do {                                                                                     \
    hipError_t e_ = (expr);                                                                \
    if (e_ != hipSuccess) {                                                                \
      set_error("fc3d_hip_mlp_create: %s -> %s", #expr, hipGetErrorString(e_));            \
      return fail(NUMERICS_ERR_DEVICE);                                                    \
    }                                                                                      \
  } while (0)
  MLP_TRY(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
  MLP_TRY(hipMalloc(&m->p, sizeof(float) * NPARAM));
  MLP_TRY(hipMalloc(&m->g, sizeof(float) * NPARAM));
  MLP_TRY(hipMalloc(&m->m1, sizeof(float) * NPARAM));
  MLP_TRY(hipMalloc(&m->m2, sizeof(float) * NPARAM));
  MLP_TRY(hipMalloc(&m->mean, sizeof(float) * MLP_NF));
  MLP_TRY(hipMalloc(&m->stdv, sizeof(float) * MLP_NF));
  for (int k = 0; k < 4; k++) {
    MLP_TRY(hipMalloc(&m->w[k], sizeof(bf16) * kDims[k][0] * kDims[k][1]));
    MLP_TRY(hipMalloc(&m->wt[k], sizeof(bf16) * kDims[k][0] * kDims[k][1]));
  }
  // He-uniform weights (seeded), zero biases; padded input columns and unused
  // output rows start at zero and only ever receive zero gradients
  std::vector<float> p(NPARAM, 0.f), zeros(NPARAM, 0.f);
  std::mt19937_64 gen(seed);
  for (int k = 0; k < 4; k++) {
    const int nout = kDims[k][0], kin = kDims[k][1];
    const int fan_in = k == 0 ? MLP_NF : MLP_H;
    const float a = std::sqrt(6.0f / (float)fan_in) * (k == 3 ? 0.1f : 1.0f);
    std::uniform_real_distribution<float> U(-a, a);
    for (int nn = 0; nn < nout; nn++)
      for (int kk = 0; kk < kin; kk++) {
        const bool used = (k != 0 || kk < MLP_NF) && (k != 3 || nn < MLP_NO);
        const float v = U(gen);
        p[(size_t)kWOff[k] + (size_t)nn * kin + kk] = used ? v : 0.f;
      }
  }
  std::vector<float> ones(MLP_NF, 1.f);
  MLP_TRY(hipMemcpy(m->p, p.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice));
  MLP_TRY(hipMemcpy(m->m1, zeros.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice));
  MLP_TRY(hipMemcpy(m->m2, zeros.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice));
  MLP_TRY(hipMemcpy(m->g, zeros.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice));
  MLP_TRY(hipMemcpy(m->mean, zeros.data(), sizeof(float) * MLP_NF, hipMemcpyHostToDevice));
  MLP_TRY(hipMemcpy(m->stdv, ones.data(), sizeof(float) * MLP_NF, hipMemcpyHostToDevice));
#undef MLP_TRY
  if ((rc = mlp_cast(m))) return fail(rc);
  if (hipStreamSynchronize(m->stream) != hipSuccess) return fail(NUMERICS_ERR_DEVICE);
  *out = m;
  return 0;
}

void fc3d_hip_mlp_destroy(fc3d_hip_mlp* m) {
  if (!m) return;
  hipSetDevice(m->device);
  if (m->stream) hipStreamSynchronize(m->stream);
  if (g_default_model == m) g_default_model = nullptr;
  void* ptrs[] = {m->p, m->g, m->m1, m->m2, m->mean, m->stdv};
  for (void* q : ptrs)
    if (q) hipFree(q);
  for (int k = 0; k < 4; k++) {
    hipFree(m->w[k]);
    hipFree(m->wt[k]);
  }
  free_workspace(m);
  if (m->stream) hipStreamDestroy(m->stream);
  delete m;
}

int fc3d_hip_mlp_get_params(const fc3d_hip_mlp* m, float* params, float* mean, float* stdv) {
  if (!m) return NUMERICS_ERR_NULL_POINTER;
  int rc = use_device(m->device);
  if (rc) return rc;
  FC3D_HIP_TRY(hipStreamSynchronize(m->stream));
  if (params) FC3D_HIP_TRY(hipMemcpy(params, m->p, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
  if (mean) FC3D_HIP_TRY(hipMemcpy(mean, m->mean, sizeof(float) * MLP_NF, hipMemcpyDeviceToHost));
  if (stdv) FC3D_HIP_TRY(hipMemcpy(stdv, m->stdv, sizeof(float) * MLP_NF, hipMemcpyDeviceToHost));
  return 0;
}

int fc3d_hip_mlp_set_params(fc3d_hip_mlp* m, const float* params, const float* mean,
                            const float* stdv) {
  if (!m) return NUMERICS_ERR_NULL_POINTER;
  if (stdv)
    for (int k = 0; k < MLP_NF; k++)
      if (!(stdv[k] > 0.f)) {
        set_error("fc3d_hip_mlp_set_params: standard deviation %d is not positive", k);
        return NUMERICS_ERR_INVALID_ARGUMENT;
      }
  int rc = use_device(m->device);
  if (rc) return rc;
  FC3D_HIP_TRY(hipStreamSynchronize(m->stream));
  if (params) FC3D_HIP_TRY(hipMemcpy(m->p, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice));
  if (mean) FC3D_HIP_TRY(hipMemcpy(m->mean, mean, sizeof(float) * MLP_NF, hipMemcpyHostToDevice));
  if (stdv) FC3D_HIP_TRY(hipMemcpy(m->stdv, stdv, sizeof(float) * MLP_NF, hipMemcpyHostToDevice));
  if ((rc = mlp_cast(m))) return rc;
  FC3D_HIP_TRY(hipStreamSynchronize(m->stream));
  return 0;
}

int fc3d_hip_mlp_forward(fc3d_hip_mlp* m, int n, const float* x, float* y) {
  if (!m || (n > 0 && (!x || !y)) || n < 0) return NUMERICS_ERR_INVALID_ARGUMENT;
  if (n == 0) return 0;
  int rc = use_device(m->device);
  if (rc) return rc;
  const size_t npad = ((size_t)n + 63) / 64 * 64;
  DevBufs B;
  float *df = nullptr, *dy = nullptr;
  bf16* dx = nullptr;
  FC3D_HIP_TRY(B.get(&df, (size_t)n * MLP_NF));
  FC3D_HIP_TRY(B.get(&dx, npad * MLP_K1));
  FC3D_HIP_TRY(B.get(&dy, (size_t)n * MLP_NO));
  FC3D_HIP_TRY(hipMemcpyAsync(df, x, sizeof(float) * (size_t)n * MLP_NF, hipMemcpyHostToDevice,
                              m->stream));
  if ((rc = mlp_forward_device(m, n, df, dx, dy, m->stream))) return rc;
  FC3D_HIP_TRY(hipMemcpyAsync(y, dy, sizeof(float) * (size_t)n * MLP_NO, hipMemcpyDeviceToHost,
                              m->stream));
  FC3D_HIP_TRY(hipStreamSynchronize(m->stream));
  return 0;
}

int fc3d_hip_mlp_gradients(fc3d_hip_mlp* m, int n, const float* x, const float* t, float* grads,
                           float* loss) {
  if (!m || !x || !t || n <= 0 || n > 65536) {
    set_error("fc3d_hip_mlp_gradients: need 1 <= n <= 65536 rows and non-NULL x, t");
    return NUMERICS_ERR_INVALID_ARGUMENT;
  }
  int rc = use_device(m->device);
  if (rc) return rc;
  const int bsz = (n + 63) / 64 * 64;
  if ((rc = mlp_workspace(m, bsz))) return rc;
  std::vector<float> tpad((size_t)bsz * MLP_NO, 0.f);
  std::memcpy(tpad.data(), t, sizeof(float) * (size_t)n * MLP_NO);
  DevBufs B;
  float *df = nullptr, *dt = nullptr;
  bf16* dx = nullptr;
  FC3D_HIP_TRY(B.get(&df, (size_t)n * MLP_NF));
  FC3D_HIP_TRY(B.get(&dx, (size_t)bsz * MLP_K1));
  FC3D_HIP_TRY(B.get(&dt, (size_t)bsz * MLP_NO));
  FC3D_HIP_TRY(hipMemcpyAsync(df, x, sizeof(float) * (size_t)n * MLP_NF, hipMemcpyHostToDevice,
                              m->stream));
  FC3D_HIP_TRY(hipMemcpyAsync(dt, tpad.data(), sizeof(float) * tpad.size(), hipMemcpyHostToDevice,
                              m->stream));
  hipLaunchKernelGGL(k_mlp_inputs, dim3((unsigned)(((size_t)bsz * MLP_K1 + 255) / 256)),
                     dim3(256), 0, m->stream, n, bsz, df, m->mean, m->stdv, dx);
  if ((rc = mlp_grad_pass(m, n, bsz, dx, dt, nullptr))) return rc;
  const double s = sum_loss(m, bsz, &rc);
  if (rc) return rc;
  if (grads) FC3D_HIP_TRY(hipMemcpy(grads, m->g, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
  if (loss) *loss = (float)(s / ((double)n * MLP_NO));
  return 0;
}

int fc3d_hip_mlp_train(fc3d_hip_mlp* m, int n, const float* x, const float* t, int epochs,
                       int batch, float lr, uint64_t seed, int set_normalisation,
                       float* final_loss) {
  if (!m || !x || !t || n <= 0 || epochs < 0 || batch < 64 || batch % 64 || !(lr > 0.f)) {
    set_error("fc3d_hip_mlp_train: invalid arguments (batch must be a positive multiple of 64)");
    return NUMERICS_ERR_INVALID_ARGUMENT;
  }
  int rc = use_device(m->device);
  if (rc) return rc;
  FC3D_HIP_TRY(hipStreamSynchronize(m->stream));
  if (set_normalisation) {
    std::vector<double> mu(MLP_NF, 0.0), var(MLP_NF, 0.0);
    for (int i = 0; i < n; i++)
      for (int k = 0; k < MLP_NF; k++) mu[(size_t)k] += x[(size_t)i * MLP_NF + k];
    for (int k = 0; k < MLP_NF; k++) mu[(size_t)k] /= n;
    for (int i = 0; i < n; i++)
      for (int k = 0; k < MLP_NF; k++) {
        const double d = x[(size_t)i * MLP_NF + k] - mu[(size_t)k];
        var[(size_t)k] += d * d;
      }
    std::vector<float> fm(MLP_NF), fs(MLP_NF);
    for (int k = 0; k < MLP_NF; k++) {
      fm[(size_t)k] = (float)mu[(size_t)k];
      const double sd = std::sqrt(var[(size_t)k] / n);
      fs[(size_t)k] = sd > 1e-6 ? (float)sd : 1.f;
    }
    FC3D_HIP_TRY(hipMemcpy(m->mean, fm.data(), sizeof(float) * MLP_NF, hipMemcpyHostToDevice));
    FC3D_HIP_TRY(hipMemcpy(m->stdv, fs.data(), sizeof(float) * MLP_NF, hipMemcpyHostToDevice));
  }
  if ((rc = mlp_workspace(m, batch))) return rc;
  DevBufs B;
  float *df = nullptr, *dt = nullptr;
  bf16* dx = nullptr;
  int* didx = nullptr;
  const int steps = std::max(1, n / batch);
  FC3D_HIP_TRY(B.get(&df, (size_t)n * MLP_NF));
  FC3D_HIP_TRY(B.get(&dx, (size_t)n * MLP_K1));
  FC3D_HIP_TRY(B.get(&dt, (size_t)n * MLP_NO));
  FC3D_HIP_TRY(B.get(&didx, (size_t)steps * batch));
  FC3D_HIP_TRY(hipMemcpyAsync(df, x, sizeof(float) * (size_t)n * MLP_NF, hipMemcpyHostToDevice,
                              m->stream));
  FC3D_HIP_TRY(hipMemcpyAsync(dt, t, sizeof(float) * (size_t)n * MLP_NO, hipMemcpyHostToDevice,
                              m->stream));
  hipLaunchKernelGGL(k_mlp_inputs, dim3((unsigned)(((size_t)n * MLP_K1 + 255) / 256)), dim3(256),
                     0, m->stream, n, n, df, m->mean, m->stdv, dx);
  std::mt19937_64 gen(seed);
  std::vector<int> perm((size_t)n), idx((size_t)steps * batch);
  for (int i = 0; i < n; i++) perm[(size_t)i] = i;
  double last = 0.0;
  const float b1 = 0.9f, b2 = 0.999f;
  for (int ep = 0; ep < epochs; ep++) {
    std::shuffle(perm.begin(), perm.end(), gen);
    for (size_t i = 0; i < idx.size(); i++) idx[i] = perm[i % (size_t)n];
    // the stream is idle here (previous epoch ended with a synchronize)
    FC3D_HIP_TRY(hipMemcpy(didx, idx.data(), sizeof(int) * idx.size(), hipMemcpyHostToDevice));
    for (int s = 0; s < steps; s++) {
      if ((rc = mlp_grad_pass(m, batch, batch, dx, dt, didx + (size_t)s * batch))) return rc;
      m->adam_t++;
      const float c1 = 1.f - (float)std::pow((double)b1, (double)m->adam_t);
      const float c2 = 1.f - (float)std::pow((double)b2, (double)m->adam_t);
      hipLaunchKernelGGL(k_adam, dim3((NPARAM + 255) / 256), dim3(256), 0, m->stream, NPARAM,
                         m->p, m->g, m->m1, m->m2, lr, b1, b2, c1, c2, 1e-8f, m->w[0], m->wt[0],
                         m->w[1], m->wt[1], m->w[2], m->wt[2], m->w[3], m->wt[3]);
      FC3D_HIP_TRY(hipGetLastError());
    }
    // the last minibatch's loss was computed with the weights before its step
    last = sum_loss(m, batch, &rc) / ((double)batch * MLP_NO);
    if (rc) return rc;
  }
  FC3D_HIP_TRY(hipStreamSynchronize(m->stream));
  if (final_loss) *final_loss = (float)last;
  return 0;
}

void fc3d_hip_set_default_model(fc3d_hip_mlp* m) { g_default_model = m; }
fc3d_hip_mlp* fc3d_hip_default_model(void) { return g_default_model; }

}  // extern "C"
