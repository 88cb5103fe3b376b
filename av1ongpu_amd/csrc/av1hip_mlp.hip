/*
 * The superblock cost model: a 24 -> 64 -> 64 -> 1 FP32 perceptron (ReLU)
 * that predicts the dependency queue's work per superblock, in microseconds,
 * from the superblock's syntax features. Training (forward, backward, Adam)
 * and inference are hand-written kernels; the decoder uses the predictions
 * only to order its queue, so pixels do not depend on them.
 *
 * Parameters, 5825 floats: W1[64][24], b1[64], W2[64][64], b2[64], W3[64],
 * b3. Features are standardised with the training set's mean and deviation;
 * the output is the standardised time.
 *
 * No counterpart in the reference: its scheduler orders work by wave only
 * (engine.cpp:1080-1302).
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <random>
#include <vector>

#include "av1hip.h"

namespace {

constexpr int kIn = AV1H_CM_FEATURES, kH = 64;
constexpr int kW1 = 0, kB1 = kW1 + kH * kIn, kW2 = kB1 + kH, kB2 = kW2 + kH * kH, kW3 = kB2 + kH, kB3 = kW3 + kH;
constexpr int kParams = kB3 + 1;
static_assert(kParams == AV1H_CM_PARAMS, "parameter count");
constexpr int kBatch = 64; /* samples per step */
constexpr int kThreads = 256;

struct Adam {
  float lr, b1, b2, eps;
  int t0; /* steps taken before this launch */
};

typedef float f4 __attribute__((ext_vector_type(4)));

/* The matrix products run on v_mfma_f32_16x16x4_f32, full FP32: lane l gives
 * A[l % 16][k] and B[k][l % 16] for one k of its group l / 16 per step and
 * holds rows 4 (l / 16) .. + 3 of column l % 16 of the result. The k of a step
 * are free to choose as long as A and B agree: step t of a 16 wide slice takes
 * k = 4 (l / 16) + t, so a lane reads its four steps' operand as one 16 byte
 * word from a k-contiguous row. */
__device__ __forceinline__ f4 mma16(f4 a, f4 b, f4 c) {
#pragma unroll
  for (int t = 0; t < 4; ++t) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], c, 0, 0, 0);
  return c;
}
__device__ __forceinline__ f4 ld4(const float* p) { return *reinterpret_cast<const f4*>(p); }
__device__ __forceinline__ void st4(float* p, f4 v) { *reinterpret_cast<f4*>(p) = v; }
/* one 16x16 tile of A B over `slices` of 16 k: rows of both k-contiguous, `row`
 * this lane's (l % 16) first element + 4 (l / 16) */
template <int kSlices>
__device__ __forceinline__ f4 tile(const float* a, const float* b, f4 c) {
#pragma unroll
  for (int q = 0; q < kSlices; ++q) c = mma16(ld4(a + 16 * q), ld4(b + 16 * q), c);
  return c;
}
template <int kCtrl>
__device__ __forceinline__ float dppf(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, false));
}
/* the sum over a row of 16 lanes, in its last lane */
__device__ __forceinline__ float row_sum(float v) {
  v += dppf<0x111>(v);
  v += dppf<0x112>(v);
  v += dppf<0x114>(v);
  return v + dppf<0x118>(v);
}
/* the sum over the four lanes l % 16 apart by 16 */
__device__ __forceinline__ float col_sum(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

/* rows of 64 (activations, W2) and 32 floats (features with a column of ones
 * for b1) padded by four, so 16 byte reads of 16 rows spread over the banks */
constexpr int kLd = kH + 4, kLx = 36, kSteps = 1024;

struct StepLds {
  float w1[kH * kLx], w2[kH * kLd], w2t[kH * kLd];
  float h1[kH * kLd]; /* then d1 transposed */
  float h1t[kH * kLd], d2[kH * kLd], d2t[kH * kLd];
  float x[kBatch * kLx], xt[2][32 * kLd];
  float out[4 * kBatch], gw3[4 * kH], gb2[4 * kH], gb3[4];
  float w3[kH], b2[kH], y[kBatch], b3, loss[16];
};

/* The gradient of the mean squared error over all n samples: batch i of
 * kBatch samples (in `perm` order) to workgroup i % gridDim.x of 16 waves that
 * each own one 16x16 tile of every 64x64 product; a workgroup's sums go to
 * part[workgroup]. What bounds a batch is one compute unit's matrix rate (992
 * tiles of 16x16x4, 3.3 us) and its five barriers. Weights and sums stay in
 * registers or LDS, activations in LDS both ways round where a product
 * contracts them; the next batch's samples load during this one. With one
 * workgroup of 256 threads and scalar FMAs the gradient over 8192 samples took
 * 13.3 ms; now 0.36. */
__global__ __launch_bounds__(kSteps) void k_mlp_grad(const float* params, float* part, const float* X,
                                                    const float* Y, const int32_t* perm, int n, float* loss) {
  __shared__ __align__(16) StepLds L;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int ts = wave >> 2, to = wave & 3;
  /* the parameters this thread owns: W2[ow + r][iw], waves 0-7 W1[o1 + r][c1]
   * (c1 = kIn: b1), then W3, b2 and b3 one each */
  const int ow = ts * 16 + 4 * g, iw = to * 16 + col;
  const int o1 = (wave >> 1) * 16 + 4 * g, c1 = (wave & 1) * 16 + col;
  const bool has1 = wave < 8 && c1 <= kIn;
  const int p1 = c1 < kIn ? kW1 + o1 * kIn + c1 : kB1 + o1, s1 = c1 < kIn ? kIn : 1;
  const int p3 = wave == 8 ? kW3 + lane : wave == 9 ? kB2 + lane : kB3;
  const bool has3 = wave == 8 || wave == 9 || (wave == 10 && lane == 0);
  for (int i = tid; i < kH * kLx; i += kSteps) {
    const int o = i / kLx, c = i - o * kLx;
    L.w1[i] = c < kIn ? params[kW1 + o * kIn + c] : c == kIn ? params[kB1 + o] : 0.f;
  }
  for (int i = tid; i < kH * kH; i += kSteps) {
    const float w = params[kW2 + i];
    L.w2[(i >> 6) * kLd + (i & 63)] = w;
    L.w2t[(i & 63) * kLd + (i >> 6)] = w;
  }
  if (tid < kH) {
    L.w3[tid] = params[kW3 + tid];
    L.b2[tid] = params[kB2 + tid];
  }
  if (tid == 0) L.b3 = params[kB3];
  /* a batch's samples: 16 threads each, features c and c + 16 */
  const int xs = tid >> 4, xc = tid & 15;
  const int nbatch = (n + kBatch - 1) / kBatch, hop = (int)gridDim.x;
  auto row_of = [&](int b) { return b < nbatch && b * kBatch + xs < n ? perm[b * kBatch + xs] : -1; };
  float fx0, fx1, fy;
  auto fetch = [&](int row) {
    fx0 = row >= 0 ? X[(size_t)row * kIn + xc] : 0.f;
    fx1 = xc < kIn - 16 ? (row >= 0 ? X[(size_t)row * kIn + 16 + xc] : 0.f) : (xc == kIn - 16 ? 1.f : 0.f);
    fy = row >= 0 && xc == 0 ? Y[row] : 0.f;
  };
  auto stage = [&](int buf) {
    L.x[xs * kLx + xc] = fx0;
    L.x[xs * kLx + 16 + xc] = fx1;
    L.xt[buf][xc * kLd + xs] = fx0;
    L.xt[buf][(16 + xc) * kLd + xs] = fx1;
    if (xc == 0) L.y[xs] = fy;
  };
  int bi = blockIdx.x, buf = 0;
  fetch(row_of(bi));
  stage(0);
  int next_row = row_of(bi + hop);
  f4 g2 = {}, g1 = {};
  float g3 = 0.f, sq = 0.f;
  const float* arow_x = L.x + (ts * 16 + col) * kLx + 4 * g;
  const float* brow_w1 = L.w1 + (to * 16 + col) * kLx + 4 * g;
  const int arow = (ts * 16 + col) * kLd + 4 * g, brow = (to * 16 + col) * kLd + 4 * g;
  __syncthreads();
  for (; bi < nbatch; bi += hop) {
    const int nb = min(kBatch, n - bi * kBatch);
    fetch(next_row);
    next_row = row_of(bi + 2 * hop);
    /* h1 = relu(x W1^T + b1) */
    f4 h1 = tile<2>(arow_x, brow_w1, f4{});
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      h1[r] = h1[r] > 0.f ? h1[r] : 0.f;
      L.h1[(ts * 16 + 4 * g + r) * kLd + iw] = h1[r];
    }
    st4(&L.h1t[iw * kLd + ow], h1);
    __syncthreads();
    /* h2 = relu(h1 W2^T + b2), its share of the output */
    const float bias = L.b2[iw], wo = L.w3[iw];
    f4 h2 = tile<4>(L.h1 + arow, L.w2 + brow, f4{bias, bias, bias, bias});
    f4 po;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      h2[r] = h2[r] > 0.f ? h2[r] : 0.f;
      po[r] = row_sum(wo * h2[r]);
    }
    if (col == 15) st4(&L.out[to * kBatch + ow], po);
    __syncthreads();
    /* the error and its gradients at the outputs of both layers */
    f4 d3 = ld4(&L.out[ow]) + ld4(&L.out[kBatch + ow]) + ld4(&L.out[2 * kBatch + ow]) + ld4(&L.out[3 * kBatch + ow]);
    const f4 y = ld4(&L.y[ow]);
    const float scale = 2.f / (float)n, b3 = L.b3;
    f4 d2;
    float s3 = 0.f, s2 = 0.f, s0 = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float e = ow + r < nb ? d3[r] + b3 - y[r] : 0.f;
      if (to == 0 && col == 0) sq += e * e;
      d3[r] = e * scale;
      d2[r] = h2[r] > 0.f ? wo * d3[r] : 0.f;
      s3 += d3[r] * h2[r];
      s2 += d2[r];
      s0 += d3[r];
      L.d2[(ts * 16 + 4 * g + r) * kLd + iw] = d2[r];
    }
    st4(&L.d2t[iw * kLd + ow], d2);
    s3 = col_sum(s3);
    s2 = col_sum(s2);
    s0 = col_sum(s0);
    if (g == 0) {
      L.gw3[ts * kH + iw] = s3;
      L.gb2[ts * kH + iw] = s2;
      if (to == 0 && col == 0) L.gb3[ts] = s0;
    }
    __syncthreads();
    /* d1 = d2 W2 where h1 is positive; the gradient of W2 */
    f4 d1 = tile<4>(L.d2 + arow, L.w2t + brow, f4{});
#pragma unroll
    for (int r = 0; r < 4; ++r) d1[r] = h1[r] > 0.f ? d1[r] : 0.f;
    st4(&L.h1[iw * kLd + ow], d1); /* d1 transposed: h1 was last read two barriers ago */
    g2 = tile<4>(L.d2t + arow, L.h1t + brow, g2);
    __syncthreads();
    /* the gradient of W1 and b1 */
    if (wave < 8)
      g1 = tile<4>(L.h1 + ((wave >> 1) * 16 + col) * kLd + 4 * g, L.xt[buf] + c1 * kLd + 4 * g, g1);
    if (has3) {
      const float* q = wave == 8 ? L.gw3 + lane : wave == 9 ? L.gb2 + lane : L.gb3;
      const int hopq = wave == 10 ? 1 : kH;
      g3 += q[0] + q[hopq] + q[2 * hopq] + q[3 * hopq];
    }
    buf ^= 1;
    stage(buf);
    __syncthreads();
  }
  float* to_part = part + (size_t)blockIdx.x * kParams;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    to_part[kW2 + (ow + r) * kH + iw] = g2[r];
    if (has1) to_part[p1 + r * s1] = g1[r];
  }
  if (has3) to_part[p3] = g3;
  if (to == 0 && col == 0) L.loss[ts * 4 + g] = sq;
  __syncthreads();
  if (tid == 0) {
    float s = 0.f;
    for (int i = 0; i < 16; ++i) s += L.loss[i];
    loss[blockIdx.x] = s / (float)n;
  }
}

struct TrainLds {
  float w1[kH * 28], w2[kH * kLd];
  float h1[kBatch * kLd], h2[kBatch * kLd], d1[kBatch * kLd], d2[kBatch * kLd];
  float x[kBatch * 28], d3[kBatch], y[kBatch];
  float e[kBatch], sq[kBatch]; /* a batch's errors; their squares summed over the batches */
  float b1[kH], b2[kH], w3[kH], b3;
};

/* An epoch: an Adam step per batch of kBatch samples in `perm` order (gradient
 * of the batch mean), one workgroup, as the steps are a chain. Adam divides by
 * the gradients' own size, so one rounded otherwise where it is close to zero
 * moves its weight by up to the learning rate: every sum of a step is one chain of
 * FMAs in the order of its index, and the matrix cores, whose sums are grouped
 * by four, are left to the gradient and the predictions. Sixteen threads per
 * sample, four neurons each; a thread's parameters (four of one column of W2
 * and one or two others) and their moments stay in registers, operands come
 * from LDS four floats a read. What bounds a step is LDS reads and its six
 * barriers. With 256 threads and a read per product a step took 107 us; two
 * epochs over 8192 samples, host work included, 27.4 ms -> 6.1. */
__global__ __launch_bounds__(kSteps) void k_mlp_train(float* params, float* am, float* av, const float* X, const float* Y,
                                                     const int32_t* perm, int n, Adam adam, float* loss) {
  __shared__ __align__(16) TrainLds L;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, s = tid >> 4, q = tid & 15;
  for (int i = tid; i < kH * kIn; i += kSteps) L.w1[i / kIn * 28 + i % kIn] = params[kW1 + i];
  for (int i = tid; i < kH * kH; i += kSteps) L.w2[(i >> 6) * kLd + (i & 63)] = params[kW2 + i];
  if (tid < kH) {
    L.b1[tid] = params[kB1 + tid];
    L.b2[tid] = params[kB2 + tid];
    L.w3[tid] = params[kW3 + tid];
  }
  if (tid < kBatch) L.sq[tid] = 0.f;
  if (tid == 0) L.b3 = params[kB3];
  /* this thread's parameters: W2[4 wave + r][lane], W1[lane][wave], and by
   * wave W1[lane][wave + 16] (0-7), b1 (8), b2 (9), W3 (10), b3 (11, one lane) */
  int pi[6];
  float* pw[6];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    pi[r] = kW2 + (4 * wave + r) * kH + lane;
    pw[r] = L.w2 + (4 * wave + r) * kLd + lane;
  }
  pi[4] = kW1 + lane * kIn + wave;
  pw[4] = L.w1 + lane * 28 + wave;
  const bool has5 = wave < 11 || (wave == 11 && lane == 0);
  pi[5] = wave < 8 ? pi[4] + 16 : wave == 8 ? kB1 + lane : wave == 9 ? kB2 + lane : wave == 10 ? kW3 + lane : kB3;
  pw[5] = wave < 8 ? pw[4] + 16 : wave == 8 ? L.b1 + lane : wave == 9 ? L.b2 + lane : wave == 10 ? L.w3 + lane : &L.b3;
  float m[6], v[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    m[k] = am[pi[k]];
    v[k] = av[pi[k]];
  }
  /* the next step's samples load during this one */
  float fx0 = 0.f, fx1 = 0.f, fy = 0.f;
  auto fetch = [&](int base) {
    const int row = base < n && base + s < n ? perm[base + s] : -1;
    fx0 = row >= 0 ? X[(size_t)row * kIn + q] : 0.f;
    fx1 = row >= 0 && q < kIn - 16 ? X[(size_t)row * kIn + 16 + q] : 0.f;
    fy = row >= 0 && q == 0 ? Y[row] : 0.f;
  };
  fetch(0);
  int step = adam.t0;
  for (int base = 0; base < n; base += kBatch) {
    const int nb = min(kBatch, n - base);
    L.x[s * 28 + q] = fx0;
    if (q < kIn - 16) L.x[s * 28 + 16 + q] = fx1;
    if (q == 0) L.y[s] = fy;
    __syncthreads();
    fetch(base + kBatch);
    float z[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) z[j] = L.b1[q + 16 * j];
#pragma unroll
    for (int i = 0; i < kIn; i += 4) {
      const f4 x = ld4(L.x + s * 28 + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f4 w = ld4(L.w1 + (q + 16 * j) * 28 + i);
#pragma unroll
        for (int t = 0; t < 4; ++t) z[j] += w[t] * x[t];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) L.h1[s * kLd + q + 16 * j] = z[j] > 0.f ? z[j] : 0.f;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) z[j] = L.b2[q + 16 * j];
#pragma unroll 4
    for (int i = 0; i < kH; i += 4) {
      const f4 h = ld4(L.h1 + s * kLd + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f4 w = ld4(L.w2 + (q + 16 * j) * kLd + i);
#pragma unroll
        for (int t = 0; t < 4; ++t) z[j] += w[t] * h[t];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      z[j] = z[j] > 0.f ? z[j] : 0.f;
      L.h2[s * kLd + q + 16 * j] = z[j];
    }
    __syncthreads();
    if (q == 0) {
      float out = L.b3;
#pragma unroll
      for (int i = 0; i < kH; i += 4) {
        const f4 h = ld4(L.h2 + s * kLd + i), w = ld4(L.w3 + i);
#pragma unroll
        for (int t = 0; t < 4; ++t) out += w[t] * h[t];
      }
      const float e = s < nb ? out - L.y[s] : 0.f;
      L.d3[s] = e * (2.f / (float)nb);
      L.e[s] = e;
    }
    __syncthreads();
    const float e3 = L.d3[s];
#pragma unroll
    for (int j = 0; j < 4; ++j) L.d2[s * kLd + q + 16 * j] = z[j] > 0.f ? L.w3[q + 16 * j] * e3 : 0.f;
    __syncthreads();
    {
      f4 g = {};
#pragma unroll 4
      for (int o = 0; o < kH; o += 4) {
        const f4 d = ld4(L.d2 + s * kLd + o);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const f4 w = ld4(L.w2 + (o + t) * kLd + 4 * q);
#pragma unroll
          for (int r = 0; r < 4; ++r) g[r] += w[r] * d[t];
        }
      }
      const f4 h = ld4(L.h1 + s * kLd + 4 * q);
#pragma unroll
      for (int r = 0; r < 4; ++r) g[r] = h[r] > 0.f ? g[r] : 0.f;
      st4(L.d1 + s * kLd + 4 * q, g);
    }
    __syncthreads();
    float g[6] = {};
#pragma unroll 4
    for (int b = 0; b < nb; ++b) {
      const f4 d2 = ld4(L.d2 + b * kLd + 4 * wave);
      const float h = L.h1[b * kLd + lane], d1 = L.d1[b * kLd + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) g[r] += d2[r] * h;
      g[4] += d1 * L.x[b * 28 + wave];
      if (wave < 8) g[5] += d1 * L.x[b * 28 + 16 + wave];
      if (wave == 8) g[5] += d1;
      if (wave == 9) g[5] += L.d2[b * kLd + lane];
      if (wave == 10) g[5] += L.d3[b] * L.h2[b * kLd + lane];
      if (wave == 11) g[5] += L.d3[b];
    }
    if (wave == 12) L.sq[lane] += L.e[lane] * L.e[lane]; /* beside the other waves' last loop */
    ++step;
    const float c1 = 1.f - powf(adam.b1, (float)step), c2 = 1.f - powf(adam.b2, (float)step);
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      if (k == 5 && !has5) break;
      m[k] = adam.b1 * m[k] + (1.f - adam.b1) * g[k];
      v[k] = adam.b2 * v[k] + (1.f - adam.b2) * g[k] * g[k];
      const float mh = m[k] / c1;
      const float vh = v[k] / c2;
      *pw[k] -= adam.lr * mh / (sqrtf(vh) + adam.eps);
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    if (k == 5 && !has5) break;
    params[pi[k]] = *pw[k];
    am[pi[k]] = m[k];
    av[pi[k]] = v[k];
  }
  /* the loss, its 64 sums in order too: equal runs report equal losses */
  if (tid == 0) {
    f4 all = {};
    for (int b = 0; b < kBatch; b += 4) all += ld4(L.sq + b);
    *loss = (all[0] + all[1] + all[2] + all[3]) / (float)n;
  }
}

/* The gradient and the loss from the workgroups' sums. */
__global__ __launch_bounds__(kThreads) void k_mlp_sum(const float* part, const float* loss, int groups, float* grad,
                                                     float* loss_out) {
  const int p = blockIdx.x * kThreads + threadIdx.x;
  if (p < kParams) {
    float s = 0.f;
    for (int i = 0; i < groups; ++i) s += part[(size_t)i * kParams + p];
    grad[p] = s;
  }
  if (p == 0) {
    float s = 0.f;
    for (int i = 0; i < groups; ++i) s += loss[i];
    *loss_out = s;
  }
}

/* Inference, a wave per 16 samples: standardise, forward on the matrix cores
 * (k_mlp_grad's tiles, weights read from the L2 by the lanes that use them,
 * hidden activations turned through LDS), back to microseconds. One thread
 * per sample left 2040 samples on 8 compute units with 64 x 64 scalar FMAs
 * one after another: a call of 2040 samples, with the pinned staging, 76 ->
 * 26 us. */
constexpr int kInferSamples = 16;
__global__ __launch_bounds__(64) void k_mlp_infer(const float* params, const float* norm, const float* X, int n,
                                                 float* out) {
  __shared__ __align__(16) float h[kInferSamples * kLd];
  const int lane = threadIdx.x, col = lane & 15, g = lane >> 4, base = blockIdx.x * kInferSamples;
  const float* row = X + (size_t)min(base + col, n - 1) * kIn;
  /* features 4g .. of each 16 wide slice; past the last one a one for b1 */
  f4 x[2], w1[4][2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int k = 16 * q + 4 * g;
    x[q] = k < kIn ? (ld4(row + k) - ld4(norm + k)) / ld4(norm + kIn + k) : f4{k == kIn ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int o = 16 * t + col;
      w1[t][q] = k < kIn ? ld4(params + kW1 + o * kIn + k) : f4{k == kIn ? params[kB1 + o] : 0.f, 0.f, 0.f, 0.f};
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const f4 z = mma16(x[1], w1[t][1], mma16(x[0], w1[t][0], f4{}));
#pragma unroll
    for (int r = 0; r < 4; ++r) h[(4 * g + r) * kLd + 16 * t + col] = z[r] > 0.f ? z[r] : 0.f;
  }
  __syncthreads();
  f4 y = {};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int o = 16 * t + col;
    const float b = params[kB2 + o], w3 = params[kW3 + o];
    f4 z = {b, b, b, b};
#pragma unroll
    for (int q = 0; q < 4; ++q) z = mma16(ld4(h + col * kLd + 16 * q + 4 * g), ld4(params + kW2 + o * kH + 16 * q + 4 * g), z);
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] += w3 * (z[r] > 0.f ? z[r] : 0.f);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) y[r] = row_sum(y[r]);
  if (col == 15) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (base + 4 * g + r < n) out[base + 4 * g + r] = (y[r] + params[kB3]) * norm[2 * kIn + 1] + norm[2 * kIn];
  }
}
unsigned infer_groups(int64_t n) { return (unsigned)((n + kInferSamples - 1) / kInferSamples); }

}  // namespace

/* The allocation-free prediction's staging (av1h_cm_predict_noalloc): the
 * features of up to AV1H_CM_NOALLOC_MAX superblocks, then their predictions.
 * Each device holds its own copy from library load to process end; host code
 * reaches it only through the address hipGetSymbolAddress gives per device. */
static __device__ __align__(256) float scratch[AV1H_CM_NOALLOC_MAX * (AV1H_CM_FEATURES + 1)];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch[kMaxDevices] = {};

/* the scratch array's address on `device`, looked up once per device with
 * that device current (at model creation) */
int scratch_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return AV1H_ERR_INVALID;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch[device]) return AV1H_OK;
  void* ptr = nullptr;
  if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return AV1H_ERR_DEVICE;
  g_scratch[device] = static_cast<float*>(ptr);
  return AV1H_OK;
}

float* scratch_of(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return g_scratch[device];
}
}  // namespace

struct av1h_costmodel {
  int device = 0;
  hipStream_t stream = nullptr;
  float* params = nullptr; /* device */
  float* adam = nullptr;   /* m then v */
  float* norm = nullptr;   /* mean[24], std[24], y mean, y std */
  int steps = 0;
  /* pinned staging of av1h_cm_predict's features and predictions, and its
   * lock (callers may predict with one model from several threads) */
  float* pin = nullptr;
  std::mutex pin_mu;
  std::vector<float> h_norm = std::vector<float>(2 * kIn + 2, 0.f);
};

namespace {

#define CM_OK(call)                         \
  do {                                      \
    if ((call) != hipSuccess) return AV1H_ERR_DEVICE; \
  } while (0)

int upload_floats(av1h_costmodel* m, float** dst, const float* src, size_t n) {
  CM_OK(hipMalloc(dst, n * sizeof(float)));
  CM_OK(hipMemcpy(*dst, src, n * sizeof(float), hipMemcpyHostToDevice));
  return AV1H_OK;
}

}  // namespace

extern "C" {

int av1h_cm_create(int device, uint64_t seed, av1h_costmodel** out) {
  if (!out) return AV1H_ERR_INVALID;
  *out = nullptr;
  av1h_device_info d;
  const int rc = av1h_describe_device(device, &d);
  if (rc != AV1H_OK) return rc;
  av1h_costmodel* m = new av1h_costmodel;
  m->device = device;
  if (hipSetDevice(device) != hipSuccess || scratch_setup(device) != AV1H_OK ||
      hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess ||
      hipMalloc(&m->params, kParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&m->adam, 2 * kParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&m->norm, (2 * kIn + 2) * sizeof(float)) != hipSuccess ||
      hipHostMalloc(&m->pin, sizeof(float) * AV1H_CM_NOALLOC_MAX * (kIn + 1), hipHostMallocDefault) != hipSuccess) {
    av1h_cm_destroy(m);
    return AV1H_ERR_DEVICE;
  }
  /* He initialisation, zero biases */
  std::vector<float> p(kParams, 0.f);
  std::mt19937_64 rng(seed);
  std::normal_distribution<float> g1(0.f, std::sqrt(2.f / kIn)), g2(0.f, std::sqrt(2.f / kH));
  for (int i = 0; i < kH * kIn; ++i) p[kW1 + i] = g1(rng);
  for (int i = 0; i < kH * kH; ++i) p[kW2 + i] = g2(rng);
  for (int i = 0; i < kH; ++i) p[kW3 + i] = g2(rng);
  for (int k = 0; k < kIn; ++k) m->h_norm[kIn + k] = 1.f;
  m->h_norm[2 * kIn + 1] = 1.f;
  if (av1h_cm_set_params(m, p.data()) != AV1H_OK ||
      av1h_cm_set_norm(m, m->h_norm.data(), m->h_norm.data() + kIn, 0.f, 1.f) != AV1H_OK) {
    av1h_cm_destroy(m);
    return AV1H_ERR_DEVICE;
  }
  *out = m;
  return AV1H_OK;
}

void av1h_cm_destroy(av1h_costmodel* m) {
  if (!m) return;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  for (void* p : {(void*)m->params, (void*)m->adam, (void*)m->norm})
    if (p) (void)hipFree(p);
  if (m->pin) (void)hipHostFree(m->pin);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
}

int av1h_cm_set_params(av1h_costmodel* m, const float* params) {
  if (!m || !params) return AV1H_ERR_INVALID;
  (void)hipSetDevice(m->device);
  CM_OK(hipMemcpy(m->params, params, kParams * sizeof(float), hipMemcpyHostToDevice));
  CM_OK(hipMemset(m->adam, 0, 2 * kParams * sizeof(float)));
  m->steps = 0;
  return AV1H_OK;
}

int av1h_cm_get_params(av1h_costmodel* m, float* params) {
  if (!m || !params) return AV1H_ERR_INVALID;
  (void)hipSetDevice(m->device);
  CM_OK(hipMemcpy(params, m->params, kParams * sizeof(float), hipMemcpyDeviceToHost));
  return AV1H_OK;
}

int av1h_cm_set_norm(av1h_costmodel* m, const float* mean, const float* dev, float y_mean, float y_dev) {
  if (!m || !mean || !dev || !(y_dev > 0.f)) return AV1H_ERR_INVALID;
  for (int k = 0; k < kIn; ++k) {
    if (!(dev[k] > 0.f)) return AV1H_ERR_INVALID;
    m->h_norm[k] = mean[k];
    m->h_norm[kIn + k] = dev[k];
  }
  m->h_norm[2 * kIn] = y_mean;
  m->h_norm[2 * kIn + 1] = y_dev;
  (void)hipSetDevice(m->device);
  CM_OK(hipMemcpy(m->norm, m->h_norm.data(), (2 * kIn + 2) * sizeof(float), hipMemcpyHostToDevice));
  return AV1H_OK;
}

int av1h_cm_get_norm(av1h_costmodel* m, float* mean, float* dev, float* y_mean, float* y_dev) {
  if (!m) return AV1H_ERR_INVALID;
  for (int k = 0; k < kIn; ++k) {
    if (mean) mean[k] = m->h_norm[k];
    if (dev) dev[k] = m->h_norm[kIn + k];
  }
  if (y_mean) *y_mean = m->h_norm[2 * kIn];
  if (y_dev) *y_dev = m->h_norm[2 * kIn + 1];
  return AV1H_OK;
}

int av1h_cm_predict(av1h_costmodel* m, const float* features, int64_t n, float* out_us) {
  if (!m || n < 0 || (n && (!features || !out_us))) return AV1H_ERR_INVALID;
  if (n == 0) return AV1H_OK;
  (void)hipSetDevice(m->device);
  if (n <= AV1H_CM_NOALLOC_MAX) {
    /* up to several 4K frames' superblocks: the kernel reads and writes the
     * pinned staging itself (25 floats a sample over PCIe once), without the
     * two allocations and two copy commands of a larger call */
    std::lock_guard<std::mutex> lk(m->pin_mu);
    float* out = m->pin + (size_t)AV1H_CM_NOALLOC_MAX * kIn;
    std::memcpy(m->pin, features, (size_t)n * kIn * sizeof(float));
    hipLaunchKernelGGL(k_mlp_infer, dim3(infer_groups(n)), dim3(64), 0, m->stream, m->params, m->norm, m->pin, (int)n,
                       out);
    CM_OK(hipGetLastError());
    CM_OK(hipStreamSynchronize(m->stream));
    std::memcpy(out_us, out, (size_t)n * sizeof(float));
    return AV1H_OK;
  }
  float *dx = nullptr, *dy = nullptr;
  int rc = upload_floats(m, &dx, features, (size_t)n * kIn);
  if (rc == AV1H_OK && hipMalloc(&dy, (size_t)n * sizeof(float)) != hipSuccess) rc = AV1H_ERR_DEVICE;
  if (rc == AV1H_OK) {
    hipLaunchKernelGGL(k_mlp_infer, dim3(infer_groups(n)), dim3(64), 0, m->stream,
                       m->params, m->norm, dx, (int)n, dy);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(out_us, dy, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, m->stream) != hipSuccess ||
        hipStreamSynchronize(m->stream) != hipSuccess)
      rc = AV1H_ERR_DEVICE;
  }
  if (dx) (void)hipFree(dx);
  if (dy) (void)hipFree(dy);
  return rc;
}

/* av1h_cm_predict without an allocation: the features and predictions are
 * staged in the device's scratch array, set up when the model was created.
 * Calls on one device share the array, so calls that overlap there race. */
int av1h_cm_predict_noalloc(av1h_costmodel* m, const float* features, int64_t n, float* out_us) {
  if (!m || n < 0 || (n && (!features || !out_us))) return AV1H_ERR_INVALID;
  if (n > AV1H_CM_NOALLOC_MAX) return AV1H_ERR_UNSUPPORTED;
  if (n == 0) return AV1H_OK;
  (void)hipSetDevice(m->device);
  float* dx = scratch_of(m->device);
  if (!dx) return AV1H_ERR_DEVICE;
  float* dy = dx + (size_t)AV1H_CM_NOALLOC_MAX * kIn;
  CM_OK(hipMemcpyAsync(dx, features, (size_t)n * kIn * sizeof(float), hipMemcpyHostToDevice, m->stream));
  hipLaunchKernelGGL(k_mlp_infer, dim3(infer_groups(n)), dim3(64), 0, m->stream,
                     m->params, m->norm, dx, (int)n, dy);
  CM_OK(hipGetLastError());
  CM_OK(hipMemcpyAsync(out_us, dy, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, m->stream));
  CM_OK(hipStreamSynchronize(m->stream));
  return AV1H_OK;
}

/* Standardised copies of the samples, with the model's normalisation. */
static void standardise(const av1h_costmodel* m, const float* X, const float* y_us, int64_t n, std::vector<float>* xs,
                        std::vector<float>* ys) {
  xs->resize((size_t)n * kIn);
  ys->resize((size_t)n);
  for (int64_t i = 0; i < n; ++i) {
    for (int k = 0; k < kIn; ++k)
      (*xs)[(size_t)i * kIn + k] = (X[(size_t)i * kIn + k] - m->h_norm[k]) / m->h_norm[kIn + k];
    (*ys)[(size_t)i] = (y_us[i] - m->h_norm[2 * kIn]) / m->h_norm[2 * kIn + 1];
  }
}

/* The standardised samples on the device, with room for an epoch's order,
 * `groups` workgroups' gradient sums and `losses` losses: one allocation. */
struct Samples {
  float *x = nullptr, *y = nullptr, *part = nullptr, *grad = nullptr, *loss = nullptr;
  int32_t* perm = nullptr;
  void* buf = nullptr;
  ~Samples() {
    if (buf) (void)hipFree(buf);
  }
  int make(const std::vector<float>& xs, const std::vector<float>& ys, int groups, int losses) {
    const size_t n = ys.size(), pad = 64;
    auto up = [&](size_t v) { return (v + pad - 1) / pad * pad; };
    const size_t total = up(n * kIn) + 2 * up(n) + up((size_t)groups * kParams) + up(kParams) + up((size_t)losses);
    CM_OK(hipMalloc(&buf, total * sizeof(float)));
    x = static_cast<float*>(buf);
    y = x + up(n * kIn);
    perm = reinterpret_cast<int32_t*>(y + up(n));
    part = reinterpret_cast<float*>(perm + up(n));
    grad = part + up((size_t)groups * kParams);
    loss = grad + up(kParams);
    CM_OK(hipMemcpy(x, xs.data(), n * kIn * sizeof(float), hipMemcpyHostToDevice));
    CM_OK(hipMemcpy(y, ys.data(), n * sizeof(float), hipMemcpyHostToDevice));
    return AV1H_OK;
  }
};

int av1h_cm_gradients(av1h_costmodel* m, const float* features, const float* y_us, int64_t n, float* grad,
                      float* loss) {
  if (!m || !features || !y_us || n <= 0 || n > (1 << 30) || !grad) return AV1H_ERR_INVALID;
  (void)hipSetDevice(m->device);
  std::vector<float> xs, ys;
  standardise(m, features, y_us, n, &xs, &ys);
  std::vector<int32_t> perm((size_t)n);
  for (int64_t i = 0; i < n; ++i) perm[(size_t)i] = (int32_t)i;
  /* batches over the compute units (a workgroup's LDS fills one) */
  const int groups = (int)std::min<int64_t>((n + kBatch - 1) / kBatch, 256);
  Samples d;
  const int rc = d.make(xs, ys, groups, groups + 1);
  if (rc != AV1H_OK) return rc;
  CM_OK(hipMemcpy(d.perm, perm.data(), perm.size() * 4, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_mlp_grad, dim3(groups), dim3(kSteps), 0, m->stream, m->params, d.part, d.x, d.y, d.perm,
                     (int)n, d.loss);
  CM_OK(hipGetLastError());
  hipLaunchKernelGGL(k_mlp_sum, dim3((kParams + kThreads - 1) / kThreads), dim3(kThreads), 0, m->stream, d.part, d.loss,
                     groups, d.grad, d.loss + groups);
  CM_OK(hipGetLastError());
  CM_OK(hipStreamSynchronize(m->stream));
  CM_OK(hipMemcpy(grad, d.grad, kParams * sizeof(float), hipMemcpyDeviceToHost));
  if (loss) CM_OK(hipMemcpy(loss, d.loss + groups, sizeof(float), hipMemcpyDeviceToHost));
  return AV1H_OK;
}

int av1h_cm_train(av1h_costmodel* m, const float* features, const float* y_us, int64_t n, int epochs, float lr,
                  uint64_t seed, int set_norm, float* loss_per_epoch) {
  if (!m || !features || !y_us || n <= 1 || n > (1 << 30) || epochs < 1 || !(lr > 0.f)) return AV1H_ERR_INVALID;
  (void)hipSetDevice(m->device);
  if (set_norm) {
    std::vector<double> mu(kIn, 0.0), sd(kIn, 0.0);
    double ym = 0, yd = 0;
    for (int64_t i = 0; i < n; ++i) {
      for (int k = 0; k < kIn; ++k) mu[k] += features[(size_t)i * kIn + k];
      ym += y_us[i];
    }
    for (int k = 0; k < kIn; ++k) mu[k] /= (double)n;
    ym /= (double)n;
    for (int64_t i = 0; i < n; ++i) {
      for (int k = 0; k < kIn; ++k) {
        const double d = features[(size_t)i * kIn + k] - mu[k];
        sd[k] += d * d;
      }
      yd += (y_us[i] - ym) * (y_us[i] - ym);
    }
    std::vector<float> fm(kIn), fs(kIn);
    for (int k = 0; k < kIn; ++k) {
      fm[k] = (float)mu[k];
      fs[k] = (float)std::max(std::sqrt(sd[k] / (double)n), 1e-3);
    }
    const int rc = av1h_cm_set_norm(m, fm.data(), fs.data(), (float)ym, (float)std::max(std::sqrt(yd / (double)n), 1e-3));
    if (rc != AV1H_OK) return rc;
  }
  std::vector<float> xs, ys;
  standardise(m, features, y_us, n, &xs, &ys);
  Samples d;
  int rc = d.make(xs, ys, 0, epochs);
  if (rc != AV1H_OK) return rc;
  /* an epoch's order is shuffled while the one before it runs, and copied
   * behind it on the stream */
  std::vector<int32_t> perm((size_t)n);
  std::mt19937_64 rng(seed);
  int done = 0; /* epochs whose launches were queued */
  for (; done < epochs; ++done) {
    for (int64_t i = 0; i < n; ++i) perm[(size_t)i] = (int32_t)i;
    std::shuffle(perm.begin(), perm.end(), rng);
    if (hipMemcpyAsync(d.perm, perm.data(), perm.size() * 4, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
        hipStreamSynchronize(m->stream) != hipSuccess)
      break;
    const Adam a{lr, 0.9f, 0.999f, 1e-8f, m->steps};
    hipLaunchKernelGGL(k_mlp_train, dim3(1), dim3(kSteps), 0, m->stream, m->params, m->adam, m->adam + kParams, d.x,
                       d.y, d.perm, (int)n, a, d.loss + done);
    if (hipGetLastError() != hipSuccess) break;
    m->steps += (int)((n + kBatch - 1) / kBatch);
  }
  CM_OK(hipStreamSynchronize(m->stream));
  if (done < epochs) return AV1H_ERR_DEVICE;
  if (loss_per_epoch)
    CM_OK(hipMemcpy(loss_per_epoch, d.loss, (size_t)epochs * sizeof(float), hipMemcpyDeviceToHost));
  return AV1H_OK;
}

}  // extern "C"
