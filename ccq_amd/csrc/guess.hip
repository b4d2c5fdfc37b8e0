// Learned starting guess for T2: a per-amplitude MLP that maps the MP2
// amplitude's local features to the converged amplitude, trained on the
// engine's own converged amplitudes with the kernels of this file.
//
// Model.  For a T2 tuple (i, j, a, b) of a spin block, m = V / D with
// V = <ij||ab> (or <ij|ab> for the alpha-beta block) and
// D = f_ii + f_jj - f_aa - f_bb.  Features, all even under i<->j and a<->b:
//   x = ( |m| / sm,  f_ii + f_jj,  f_aa + f_bb,  V_ijij,  V_abab )
// (sm = rms of m over the block).  The network predicts r and the guess is
// t = m (1 + r), antisymmetric wherever m is and zero where m is.
// Network: x -> (x - mu) / sd -> 64 tanh -> 64 tanh -> 1, weights and layer
// inputs rounded to BF16 (round to nearest even), products accumulated in
// FP32.  Loss: mean over samples of ((m / sm) r - y)^2 with y = (t_conv - m) / sm.
//
// Training (ccq_hip_mlp_train) runs on the GPU: per step a batch of samples
// drawn by a counter-based hash, forward, backward and the workgroup's share
// of the gradient in one kernel (one lane per hidden unit), then a kernel
// that sums the workgroups' shares in a fixed order (deterministic) and does
// the Adam step.
// ccq has no counterpart (its guess is T = 0, src/calc_driver.f90:210-211).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/ccq_hip.h"
#include "kernels.h"

namespace ccqk {

constexpr int F = kGuessFeatures;
constexpr int H = kGuessHidden;
// parameter offsets
constexpr int P_MU = 0, P_SD = F, P_W1 = 2 * F, P_B1 = P_W1 + F * H, P_W2 = P_B1 + H,
              P_B2 = P_W2 + H * H, P_W3 = P_B2 + H, P_B3 = P_W3 + H;
static_assert(P_B3 + 1 == kGuessParams, "parameter layout");

// round to the nearest BF16 (ties to even), returned as float
__host__ __device__ inline float bf16r(float x) {
  uint32_t u;
  memcpy(&u, &x, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  u &= 0xFFFF0000u;
  float y;
  memcpy(&y, &u, 4);
  return y;
}

struct Tuple {
  double m;
  float x[F];
};

__device__ inline Tuple tuple_at(const GuessBlock& B, int64_t i, int64_t j, int64_t a, int64_t b) {
  const int64_t nc = B.nc, nc2 = nc * nc, nc3 = nc2 * nc;
  const int64_t A = B.va0 + a, Bv = B.vb0 + b;
  const double V = B.V[i * nc3 + j * nc2 + A * nc + Bv];
  const double so = B.f1[i] + B.f2[j];
  const double sv = B.f1[B.o1 + a] + B.f2[B.o2 + b];
  Tuple t;
  t.m = V / (so - sv);
  t.x[0] = (float)(fabs(t.m) * B.inv_sm);
  t.x[1] = (float)so;
  t.x[2] = (float)sv;
  t.x[3] = (float)B.V[i * nc3 + j * nc2 + i * nc + j];
  t.x[4] = (float)B.V[A * nc3 + Bv * nc2 + A * nc + Bv];
  return t;
}

__device__ inline Tuple guess_tuple(const GuessBlock& B, int64_t e, int64_t& off) {
  int64_t r = e;
  const int64_t b = r % B.v2; r /= B.v2;
  const int64_t a = r % B.v1; r /= B.v1;
  const int64_t j = r % B.o2; r /= B.o2;
  const int64_t i = r;
  off = e;
  return tuple_at(B, i, j, a, b);
}

// p-th pair (x < y) of n in row order (0,1), (0,2), ..., (1,2), ...
__device__ inline void pair_of(int64_t p, int64_t n, int64_t& x, int64_t& y) {
  const int64_t total = n * (n - 1) / 2;
  const int64_t q = total - 1 - p;   // pairs counted from the end
  int64_t k = (int64_t)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
  while ((k + 1) * (k + 2) / 2 <= q) ++k;
  while (k * (k + 1) / 2 > q) --k;
  x = n - 2 - k;
  y = n - 1 - (q - k * (k + 1) / 2);
}

__global__ __launch_bounds__(256) void guess_msq(GuessBlock B, double* __restrict__ partial) {
  __shared__ double red[256];
  const int64_t total = B.o1 * B.o2 * B.v1 * B.v2;
  double acc = 0.0;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    int64_t off;
    const Tuple t = guess_tuple(B, e, off);
    acc += t.m * t.m;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// weights into LDS, BF16-rounded (mu, sd and biases are kept in FP32)
__device__ inline void load_weights(float* w, const float* __restrict__ params) {
  for (int k = threadIdx.x; k < kGuessParams; k += blockDim.x) {
    const bool wt = (k >= P_W1 && k < P_B1) || (k >= P_W2 && k < P_B2) || (k >= P_W3 && k < P_B3);
    w[k] = wt ? bf16r(params[k]) : params[k];
  }
  __syncthreads();
}

// Inference of one sample per thread, with the first hidden layer in LDS
// (hs: this thread's column, stride kApplyThreads) instead of a per-thread
// array, which the run-time indexed loops would otherwise place in scratch
// memory.  Every sum runs in index order, as in mlp_step.
constexpr int kApplyThreads = 128;
__device__ inline float mlp_infer(const float* __restrict__ w, const float (&xin)[F], float* hs) {
  float x[F];
#pragma unroll
  for (int k = 0; k < F; ++k) x[k] = bf16r((xin[k] - w[P_MU + k]) / w[P_SD + k]);
#pragma unroll 8
  for (int p = 0; p < H; ++p) {
    float acc = w[P_B1 + p];
#pragma unroll
    for (int k = 0; k < F; ++k) acc += w[P_W1 + k * H + p] * x[k];
    hs[p * kApplyThreads] = bf16r(tanhf(acc));
  }
  float out = w[P_B3];
  for (int q = 0; q < H; ++q) {
    float acc = w[P_B2 + q];
#pragma unroll 16
    for (int p = 0; p < H; ++p) acc += w[P_W2 + p * H + q] * hs[p * kApplyThreads];
    out += w[P_W3 + q] * bf16r(tanhf(acc));
  }
  return out;
}

__global__ __launch_bounds__(kApplyThreads) void guess_apply(GuessBlock B, const float* __restrict__ params) {
  __shared__ float w[kGuessParams];
  __shared__ float h1s[H * kApplyThreads];
  float* hs = h1s + threadIdx.x;
  if (params) load_weights(w, params);
  if (B.anti) {
    // t[ijab] = -t[jiab] = -t[ijba] = t[jiba]; the network sees features
    // that are even under both swaps, so one evaluation serves all four
    const int64_t po = B.o1 * (B.o1 - 1) / 2, pv = B.v1 * (B.v1 - 1) / 2;
    const int64_t total = po * pv;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
      int64_t i, j, a, b;
      pair_of(e / pv, B.o1, i, j);
      pair_of(e % pv, B.v1, a, b);
      const Tuple t = tuple_at(B, i, j, a, b);
      double v = t.m;
      if (params) v = t.m * (1.0 + (double)mlp_infer(w, t.x, hs));
      const int64_t o = B.o2, vv = B.v2;
      B.t[((i * o + j) * B.v1 + a) * vv + b] = v;
      B.t[((j * o + i) * B.v1 + a) * vv + b] = -v;
      B.t[((i * o + j) * B.v1 + b) * vv + a] = -v;
      B.t[((j * o + i) * B.v1 + b) * vv + a] = v;
    }
    return;
  }
  const int64_t total = B.o1 * B.o2 * B.v1 * B.v2;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    int64_t off;
    const Tuple t = guess_tuple(B, e, off);
    double v = t.m;
    if (params) v = t.m * (1.0 + (double)mlp_infer(w, t.x, hs));
    B.t[off] = v;
  }
}

__global__ __launch_bounds__(256) void guess_data(GuessBlock B, float* __restrict__ X,
                                                  float* __restrict__ M, float* __restrict__ Y) {
  const int64_t total = B.o1 * B.o2 * B.v1 * B.v2;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    int64_t off;
    const Tuple t = guess_tuple(B, e, off);
#pragma unroll
    for (int k = 0; k < F; ++k) X[e * F + k] = t.x[k];
    M[e] = (float)(t.m * B.inv_sm);
    Y[e] = (float)((B.t[off] - t.m) * B.inv_sm);
  }
}

static int grid_of(int64_t n) {
  int64_t g = (n + 255) / 256;
  return (int)(g < 1 ? 1 : (g > 4096 ? 4096 : g));
}

hipError_t launch_guess_msq(hipStream_t s, const GuessBlock& B, double* partial, int blocks) {
  hipLaunchKernelGGL(guess_msq, dim3(blocks), dim3(256), 0, s, B, partial);
  return hipGetLastError();
}

hipError_t launch_guess_apply(hipStream_t s, const GuessBlock& B, const float* params) {
  if (B.anti && (B.o1 != B.o2 || B.v1 != B.v2 || B.va0 != B.vb0 || B.f1 != B.f2))
    return hipErrorInvalidValue;
  const int64_t total = B.anti ? (B.o1 * (B.o1 - 1) / 2) * (B.v1 * (B.v1 - 1) / 2)
                               : B.o1 * B.o2 * B.v1 * B.v2;
  if (total <= 0) return hipSuccess;
  const int64_t blocks = (total + kApplyThreads - 1) / kApplyThreads;
  hipLaunchKernelGGL(guess_apply, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(kApplyThreads), 0, s, B,
                     params);
  return hipGetLastError();
}

hipError_t launch_guess_data(hipStream_t s, const GuessBlock& B, float* X, float* M, float* Y) {
  const int64_t total = B.o1 * B.o2 * B.v1 * B.v2;
  if (total <= 0) return hipSuccess;
  hipLaunchKernelGGL(guess_data, dim3(grid_of(total)), dim3(256), 0, s, B, X, M, Y);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// training

__device__ inline uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Forward, backward and gradient of kStepTile samples at a time per workgroup.
// A lane is a hidden unit and a wave carries four samples, so the 64-long sums
// read the weights once per four samples, the activations stay in LDS, and
// 4096 samples fill 256 workgroups (a thread per sample filled 16).  The
// gradient is the outer product of activations and signals: a thread owns a
// 4 x 4 tile of W2 and up to three of the other entries, in FP64; each
// workgroup stores its share (partial[block][k]) and mlp_reduce sums them.
// Bound by the latency of the six phases.  Batch 4096: 275 us (a thread per
// sample, activations through memory) + 1687 us (a thread per parameter,
// serial over the batch) before, 22 us + 5.7 us (mlp_reduce) now.
constexpr int kStepThreads = 256;
constexpr int kStepTile = 16;       // samples of one pass
constexpr int kStepBlocks = 256;    // most workgroups (one pass each at batch 4096)
constexpr int kW2P = H + 1;         // W2 rows and columns both read without bank conflicts
constexpr int kActP = H + 4;        // row pitch of the samples' activations, 16-byte aligned
constexpr int kGradN = kGuessParams + 1;   // gradient and loss (mu, sd entries unused)
constexpr int kExtra = (kGradN - P_W1 - H * H + kStepThreads - 1) / kStepThreads;

// gradient entry k as sum_s act[s][a] * sig[s][b]; columns of a sample's row:
// x (F), 1, h1, h2, gh1, gh2, g, e^2
constexpr int C_X = 0, C_ONE = F, C_H1 = 8, C_H2 = C_H1 + kActP, C_G1 = C_H2 + kActP, C_G2 = C_G1 + kActP,
              C_G = C_G2 + kActP, C_E = C_G + 1, kRow = C_G + 4;
__device__ inline void grad_columns(int k, int& a, int& b) {
  if (k < P_B1) {
    a = C_X + (k - P_W1) / H;
    b = C_G1 + (k - P_W1) % H;
  } else if (k < P_W2) {
    a = C_ONE;
    b = C_G1 + (k - P_B1);
  } else if (k < P_W3) {
    a = C_ONE;
    b = C_G2 + (k - P_B2);
  } else if (k < P_B3) {
    a = C_H2 + (k - P_W3);
    b = C_G;
  } else {
    a = C_ONE;
    b = k == P_B3 ? C_G : C_E;
  }
}

__global__ __launch_bounds__(kStepThreads) void mlp_step(const float* __restrict__ params,
                                                         const float* __restrict__ X,
                                                         const float* __restrict__ Mv,
                                                         const float* __restrict__ Yv, int64_t n,
                                                         int64_t batch, uint64_t seed, int64_t step, int full,
                                                         double* __restrict__ partial) {
  __shared__ __align__(16) float rows[kStepTile * kRow];
  __shared__ float w2[H * kW2P];
  __shared__ float w[kGuessParams - H * H];   // the other parameters, in order
  auto at = [](int k) { return k < P_W2 ? k : k - H * H; };
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int k = tid; k < kGuessParams; k += kStepThreads) {
    const bool wt = (k >= P_W1 && k < P_B1) || (k >= P_W2 && k < P_B2) || (k >= P_W3 && k < P_B3);
    const float v = wt ? bf16r(params[k]) : params[k];
    if (k >= P_W2 && k < P_B2) w2[(k - P_W2) / H * kW2P + (k - P_W2) % H] = v;
    else w[at(k)] = v;
  }
  const int p0 = (tid >> 4) * 4, q0 = (tid & 15) * 4;
  double acc[4][4], ext[kExtra];
  int ea[kExtra], eb[kExtra];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0;
#pragma unroll
  for (int x = 0; x < kExtra; ++x) {
    ext[x] = 0.0;
    // entry number tid + x kStepThreads of those outside W2
    const int e = P_W1 + tid + x * kStepThreads;
    const int k = e < P_W2 ? e : e + H * H;
    ea[x] = eb[x] = -1;
    if (k < kGradN) grad_columns(k, ea[x], eb[x]);
  }

  for (int64_t s0 = (int64_t)blockIdx.x * kStepTile; s0 < batch; s0 += (int64_t)gridDim.x * kStepTile) {
    auto sample = [&](int s) -> int64_t {
      return full ? s0 + s : (int64_t)(mix64(seed ^ mix64((uint64_t)step * 0x100000001ull + (uint64_t)(s0 + s))) %
                                       (uint64_t)n);
    };
    __syncthreads();   // the weights are in; the previous pass's rows are read
    if (tid < kStepTile * F) {
      const int s = tid / F, k = tid % F;
      float x = 0.0f;
      if (s0 + s < batch) x = bf16r((X[sample(s) * F + k] - w[P_MU + k]) / w[P_SD + k]);
      rows[s * kRow + C_X + k] = x;
      if (k == 0) rows[s * kRow + C_ONE] = 1.0f;
    }
    __syncthreads();
    float* r0 = rows + wave * 4 * kRow;   // this wave's four samples
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float* r = r0 + i * kRow;
      float a = w[P_B1 + lane];
#pragma unroll
      for (int k = 0; k < F; ++k) a += w[P_W1 + k * H + lane] * r[C_X + k];
      r[C_H1 + lane] = bf16r(tanhf(a));
    }
    __syncthreads();
    {
      float a[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = w[at(P_B2) + lane];
#pragma unroll 4
      for (int p = 0; p < H; p += 4) {
        float4 h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = *reinterpret_cast<const float4*>(r0 + i * kRow + C_H1 + p);
        const float u0 = w2[p * kW2P + lane], u1 = w2[(p + 1) * kW2P + lane], u2 = w2[(p + 2) * kW2P + lane],
                    u3 = w2[(p + 3) * kW2P + lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a[i] += u0 * h[i].x;
          a[i] += u1 * h[i].y;
          a[i] += u2 * h[i].z;
          a[i] += u3 * h[i].w;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) r0[i * kRow + C_H2 + lane] = bf16r(tanhf(a[i]));
    }
    __syncthreads();
    if (tid < kStepTile) {
      float* r = rows + tid * kRow;
      float out = w[at(P_B3)];
      for (int q = 0; q < H; ++q) out += w[at(P_W3) + q] * r[C_H2 + q];
      float g = 0.0f, e2 = 0.0f;
      if (s0 + tid < batch) {
        const int64_t idx = sample(tid);
        const float mm = Mv[idx];
        const float e = mm * out - Yv[idx];
        g = 2.0f * e * mm / (float)batch;
        e2 = e * e;
      }
      r[C_G] = g;
      r[C_E] = e2;
    }
    __syncthreads();
    // gh2 = g W3 (1 - h2^2); gh1 = (W2 gh2) (1 - h1^2)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float* r = r0 + i * kRow;
      const float h2 = r[C_H2 + lane];
      r[C_G2 + lane] = r[C_G] * w[at(P_W3) + lane] * (1.0f - h2 * h2);
    }
    __syncthreads();
    {
      float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
      for (int q = 0; q < H; q += 4) {
        float4 h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = *reinterpret_cast<const float4*>(r0 + i * kRow + C_G2 + q);
        const float* u = w2 + lane * kW2P + q;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a[i] += u[0] * h[i].x;
          a[i] += u[1] * h[i].y;
          a[i] += u[2] * h[i].z;
          a[i] += u[3] * h[i].w;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float* r = r0 + i * kRow;
        const float h1 = r[C_H1 + lane];
        r[C_G1 + lane] = a[i] * (1.0f - h1 * h1);
      }
    }
    __syncthreads();
    auto add = [&](int s) {
      const float* r = rows + s * kRow;
      const float4 h = *reinterpret_cast<const float4*>(r + C_H1 + p0);
      const float4 g = *reinterpret_cast<const float4*>(r + C_G2 + q0);
      const double hd[4] = {h.x, h.y, h.z, h.w}, gd[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += hd[i] * gd[j];
#pragma unroll
      for (int x = 0; x < kExtra; ++x)
        if (ea[x] >= 0) ext[x] += (double)r[ea[x]] * (double)r[eb[x]];
    };
    // (rows past the batch are left out, not weighted by zero: with infinite
    // weights they hold NaN; a full pass keeps its constant length: 25 steps of
    // 4096 samples 1009 us, with the run-time one 1027)
    if (batch - s0 >= kStepTile)
      for (int s = 0; s < kStepTile; ++s) add(s);
    else
      for (int s = 0; s < (int)(batch - s0); ++s) add(s);
  }

  double* out = partial + (int64_t)blockIdx.x * kGradN;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) out[P_W2 + (p0 + i) * H + q0 + j] = acc[i][j];
#pragma unroll
  for (int x = 0; x < kExtra; ++x) {
    const int e = P_W1 + tid + x * kStepThreads;
    const int k = e < P_W2 ? e : e + H * H;
    if (k < kGradN) out[k] = ext[x];
  }
}

// workgroups of mlp_step for a batch
static int step_blocks(int64_t batch) {
  const int64_t b = (batch + kStepTile - 1) / kStepTile;
  return (int)(b < kStepBlocks ? b : kStepBlocks);
}

// grad[k] = sum over the workgroups' shares in order (mu / sd get 0),
// grad[kGuessParams] = loss; with adam set, the Adam step of that gradient.
// A lane per entry, the shares in four runs (one per wave) added in order.
__global__ __launch_bounds__(256) void mlp_reduce(const double* __restrict__ partial, int blocks, int64_t batch,
                                                  float* __restrict__ grad, int adam, float* __restrict__ params,
                                                  float* __restrict__ m1, float* __restrict__ m2, float lr, float c1,
                                                  float c2) {
  __shared__ double red[3][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int k = blockIdx.x * 64 + lane;
  const int per = (blocks + 3) / 4, lo = wave * per, hi = lo + per < blocks ? lo + per : blocks;
  double acc = 0.0;
  if (k >= P_W1 && k < kGradN) {
#pragma unroll 8
    for (int b = lo; b < hi; ++b) acc += partial[(int64_t)b * kGradN + k];
  }
  if (wave) red[wave - 1][lane] = acc;
  __syncthreads();
  if (wave || k >= kGradN) return;
  acc = ((acc + red[0][lane]) + red[1][lane]) + red[2][lane];
  const float g = (float)(k == kGuessParams ? acc / (double)batch : acc);
  grad[k] = g;
  if (!adam || k < P_W1 || k >= kGuessParams) return;
  const float a = 0.9f * m1[k] + 0.1f * g, b = 0.999f * m2[k] + 0.001f * g * g;
  m1[k] = a;
  m2[k] = b;
  params[k] -= lr * (a / c1) / (sqrtf(b / c2) + 1e-8f);
}

}  // namespace ccqk

// ---------------------------------------------------------------------------
// C ABI (standalone: device-resident training data, one GPU)

namespace {

thread_local std::string g_guess_err;

struct DevF {
  float* p = nullptr;
  explicit DevF(int64_t n) {
    if (hipMalloc(&p, sizeof(float) * (n > 0 ? n : 1)) != hipSuccess) p = nullptr;
  }
  ~DevF() {
    if (p) (void)hipFree(p);
  }
};

#define GCHK(x)                                                            \
  do {                                                                     \
    hipError_t e_ = (x);                                                   \
    if (e_ != hipSuccess) {                                                \
      g_guess_err = std::string(#x) + ": " + hipGetErrorString(e_);        \
      return 1;                                                            \
    }                                                                      \
  } while (0)

// loss and gradient of one batch (device buffers; partial holds
// step_blocks(batch) * kGradN doubles, grad kGradN floats), on the null stream;
// full: the batch is samples 0 .. batch - 1, else drawn by (seed, step).  With
// m1, the Adam step of that gradient follows (bias corrections c1, c2).
hipError_t launch_step(float* P, const float* X, const float* M, const float* Y, int64_t n, int64_t batch,
                       uint64_t seed, int64_t step, int full, double* partial, float* grad, float* m1 = nullptr,
                       float* m2 = nullptr, float lr = 0.0f, float c1 = 1.0f, float c2 = 1.0f) {
  using namespace ccqk;
  const int blocks = step_blocks(batch);
  hipLaunchKernelGGL(mlp_step, dim3(blocks), dim3(kStepThreads), 0, 0, P, X, M, Y, n, batch, seed, step, full,
                     partial);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(mlp_reduce, dim3((kGradN + 63) / 64), dim3(256), 0, 0, partial, blocks, batch, grad,
                     m1 ? 1 : 0, P, m1, m2, lr, c1, c2);
  return hipGetLastError();
}

int run_training(const float* X, const float* M, const float* Y, int64_t n, float* params,
                 int64_t nparams, int64_t steps, int64_t batch, double lr, uint64_t seed,
                 double* loss_out, float* grad_out) {
  using namespace ccqk;
  if (nparams != kGuessParams) {
    g_guess_err = "nparams must be " + std::to_string(kGuessParams);
    return 2;
  }
  if (n <= 0 || batch <= 0 || (grad_out && batch != n)) {
    g_guess_err = "bad sample / batch count";
    return 2;
  }
  DevF dX(n * F), dM(n), dY(n), dP(kGuessParams), dG(kGradN), dm1(kGuessParams), dm2(kGuessParams),
      dS((int64_t)2 * step_blocks(batch) * kGradN);
  double* part = reinterpret_cast<double*>(dS.p);
  if (!dX.p || !dM.p || !dY.p || !dP.p || !dG.p || !dm1.p || !dm2.p || !dS.p) {
    g_guess_err = "out of device memory";
    return 1;
  }
  GCHK(hipMemcpy(dX.p, X, sizeof(float) * n * F, hipMemcpyHostToDevice));
  GCHK(hipMemcpy(dM.p, M, sizeof(float) * n, hipMemcpyHostToDevice));
  GCHK(hipMemcpy(dY.p, Y, sizeof(float) * n, hipMemcpyHostToDevice));
  GCHK(hipMemcpy(dP.p, params, sizeof(float) * kGuessParams, hipMemcpyHostToDevice));
  GCHK(hipMemset(dm1.p, 0, sizeof(float) * kGuessParams));
  GCHK(hipMemset(dm2.p, 0, sizeof(float) * kGuessParams));
  if (grad_out) {
    GCHK(launch_step(dP.p, dX.p, dM.p, dY.p, n, n, 0, 0, 1, part, dG.p));
    steps = 0;
  }
  double b1 = 1.0, b2 = 1.0;
  for (int64_t st = 0; st < steps; ++st) {
    b1 *= 0.9;
    b2 *= 0.999;
    GCHK(launch_step(dP.p, dX.p, dM.p, dY.p, n, batch, seed, st, 0, part, dG.p, dm1.p, dm2.p, (float)lr,
                     (float)(1.0 - b1), (float)(1.0 - b2)));
  }
  float loss = 0.0f;
  GCHK(hipMemcpy(&loss, dG.p + kGuessParams, sizeof(float), hipMemcpyDeviceToHost));
  if (loss_out) *loss_out = loss;
  if (grad_out) GCHK(hipMemcpy(grad_out, dG.p, sizeof(float) * kGuessParams, hipMemcpyDeviceToHost));
  else GCHK(hipMemcpy(params, dP.p, sizeof(float) * kGuessParams, hipMemcpyDeviceToHost));
  GCHK(hipDeviceSynchronize());
  return 0;
}

// ---------------------------------------------------------------------------
// Gradient without device allocation: every device buffer of the gradient
// (the staged samples and parameters, the workgroups' shares, the gradient
// and loss) lives in one file-scope array.  Each GPU
// holds its own copy until the process ends; its address is looked up once
// per device and used for every kernel argument and copy.

constexpr int64_t kNaMax = CCQ_HIP_MLP_NOALLOC_MAX_SAMPLES;
constexpr int64_t kNaX = 0;                                   // X[n][F]
constexpr int64_t kNaM = kNaX + kNaMax * ccqk::F;             // M[n]
constexpr int64_t kNaY = kNaM + kNaMax;                       // Y[n]
constexpr int64_t kNaP = kNaY + kNaMax;                       // params
constexpr int64_t kNaG = kNaP + 64 * ((ccqk::kGuessParams + 63) / 64);        // grad + loss
constexpr int64_t kNaS = kNaG + 64 * ((ccqk::kGradN + 63) / 64);              // shares (doubles)
constexpr int64_t kNaFloats = kNaS + 2 * (int64_t)ccqk::kStepBlocks * ccqk::kGradN;

constexpr int kNaDevices = 64;
std::mutex g_na_mu;
float* g_na_ptr[kNaDevices] = {};

}  // namespace

static __device__ __align__(256) float scratch[kNaFloats];

namespace {

// the device address of this GPU's scratch (looked up on first use)
float* noalloc_scratch(int dev) {
  std::lock_guard<std::mutex> lk(g_na_mu);
  if (!g_na_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      g_guess_err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
      return nullptr;
    }
    g_na_ptr[dev] = static_cast<float*>(p);
  }
  return g_na_ptr[dev];
}

}  // namespace

extern "C" {

int ccq_hip_mlp_grad_noalloc(const float* X, const float* M, const float* Y, int64_t n,
                             const float* params, int64_t nparams, float* grad, double* loss) {
  using namespace ccqk;
  if (nparams != kGuessParams) {
    g_guess_err = "nparams must be " + std::to_string(kGuessParams);
    return 2;
  }
  if (n <= 0 || n > kNaMax) {
    g_guess_err = "sample count must be in 1.." + std::to_string(kNaMax) +
                  " (CCQ_HIP_MLP_NOALLOC_MAX_SAMPLES) for ccq_hip_mlp_grad_noalloc";
    return 2;
  }
  if (!X || !M || !Y || !params || !grad) {
    g_guess_err = "null array";
    return 2;
  }
  int dev = 0;
  GCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kNaDevices) {
    g_guess_err = "device ordinal beyond the scratch table";
    return 2;
  }
  float* s = noalloc_scratch(dev);
  if (!s) return 1;
  GCHK(hipMemcpy(s + kNaX, X, sizeof(float) * n * F, hipMemcpyHostToDevice));
  GCHK(hipMemcpy(s + kNaM, M, sizeof(float) * n, hipMemcpyHostToDevice));
  GCHK(hipMemcpy(s + kNaY, Y, sizeof(float) * n, hipMemcpyHostToDevice));
  GCHK(hipMemcpy(s + kNaP, params, sizeof(float) * kGuessParams, hipMemcpyHostToDevice));
  GCHK(launch_step(s + kNaP, s + kNaX, s + kNaM, s + kNaY, n, n, 0, 0, 1, reinterpret_cast<double*>(s + kNaS),
                   s + kNaG));
  float l = 0.0f;
  GCHK(hipMemcpy(&l, s + kNaG + kGuessParams, sizeof(float), hipMemcpyDeviceToHost));
  GCHK(hipMemcpy(grad, s + kNaG, sizeof(float) * kGuessParams, hipMemcpyDeviceToHost));
  GCHK(hipDeviceSynchronize());
  if (loss) *loss = l;
  return 0;
}

int64_t ccq_hip_mlp_nparams(void) { return ccqk::kGuessParams; }

int ccq_hip_mlp_train(const float* X, const float* M, const float* Y, int64_t n, float* params,
                      int64_t nparams, int64_t steps, int64_t batch, double lr, uint64_t seed,
                      double* final_loss) {
  return run_training(X, M, Y, n, params, nparams, steps, batch, lr, seed, final_loss, nullptr);
}

int ccq_hip_mlp_grad(const float* X, const float* M, const float* Y, int64_t n, const float* params,
                     int64_t nparams, float* grad, double* loss) {
  std::vector<float> p(params, params + (nparams > 0 ? nparams : 0));
  return run_training(X, M, Y, n, p.data(), nparams, 1, n, 0.0, 0, loss, grad);
}

const char* ccq_hip_mlp_last_error(void) { return g_guess_err.c_str(); }

}  // extern "C"
