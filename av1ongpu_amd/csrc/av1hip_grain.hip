/*
 * Film grain synthesis (specification 7.18.3) on gfx950.
 *
 * The reference synthesises the grain on the host every frame and uploads a
 * full-frame noise image (src/core/grain.cpp:70-139, 6.2 MB at 1080p). Here the
 * three grain templates (82x73 luma, 44x38 chroma at 4:2:0) and the per stripe
 * block offsets are built on a second stream (k_grain_template,
 * av1hip_grain_template.hpp), and
 *   k_grain_apply - the noise sample of every picture sample is derived on
 *     the fly from the templates (the block and stripe overlap blends of
 *     av1gpu_kernels.h:3218-3291 evaluated per sample) and blended in, chroma
 *     before luma inside each tile because chroma reads the luma before grain.
 * The arithmetic is the reference's (av1gpu_kernels.h:3039-3365).
 */
#define AV1T_TABLE_QUAL static __constant__ const
#include "av1hip_grain_template.hpp"
#include "spec_tables.h"

namespace av1hip {
namespace {

#define SPEC(off) (av1t_spec_table + (off))

constexpr int kLW = 82, kLH = 73;

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }
__device__ __forceinline__ int grnd(int v, int n) { return n <= 0 ? v : (v + (1 << (n - 1))) >> n; }

/* two workgroups (of one wave) per frame with film grain, a half each */
__global__ __launch_bounds__(64) void k_grain_template(BatchDev B) {
  __shared__ __align__(16) uint8_t s_lds[grain::kTemplateLds];
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKGrainTemplate);
  const int total = pre[B.njobs];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int j = find_job(pre, B.njobs, v);
    grain::template_half(filter_args(B, j), v - pre[j], s_lds);
    __syncthreads();
  }
}

struct NoiseCtx {
  const int16_t* t;   /* template of this plane */
  const uint8_t* offs;
  int tw, blocks, sx, sy, overlap, lo, hi;
  __device__ __forceinline__ int G(int s, int b, int i, int j) const {
    const int r = offs[s * blocks + b];
    const int ox = r >> 4, oy = r & 15;
    const int gx = sx ? 6 + ox : 9 + 2 * ox, gy = sy ? 6 + oy : 9 + 2 * oy;
    return t[(gy + i) * tw + gx + j];
  }
  /* the stripe buffer after the horizontal overlap blends */
  __device__ __forceinline__ int H(int s, int i, int x) const {
    const int lbw = 5 - sx, bw = 1 << lbw;
    const int b = x >> lbw, j = x & (bw - 1);
    int g = G(s, b, i, j);
    if (overlap && b > 0 && j < (sx ? 1 : 2)) {
      const int old = G(s, b - 1, i, j + bw);
      g = clampi(grnd(sx ? old * 23 + g * 22 : (j == 0 ? old * 27 + g * 17 : old * 17 + g * 27), 5), lo, hi);
    }
    return g;
  }
  /* the noise image sample after the vertical blends */
  __device__ __forceinline__ int N(int x, int y) const {
    const int lbh = 5 - sy, bh = 1 << lbh;
    const int s = y >> lbh, row = y & (bh - 1);
    int v = H(s, row, x);
    if (overlap && s > 0 && row < (sy ? 1 : 2)) {
      const int old = H(s - 1, row + bh, x);
      v = clampi(grnd(sy ? old * 23 + v * 22 : (row == 0 ? old * 27 + v * 17 : old * 17 + v * 27), 5), lo, hi);
    }
    return v;
  }
};

__device__ __forceinline__ int scale_lut(const int* lut, int index, int bd) {
  const int sh = bd - 8;
  const int x = sh > 0 ? index >> sh : index;
  if (bd == 8 || x >= 255) return lut[x > 255 ? 255 : x];
  const int rem = index - (x << sh);
  return lut[x] + grnd((lut[x + 1] - lut[x]) * rem, sh);
}

/* 64x32 luma tiles (32x16 chroma at 4:2:0), 256 threads */
__device__ void grain_tile(FArgs a, int t, int* s_lut) {
  LayRef L = a.lay;
  const DevGrain& g = *a.plan.grain;
  const int16_t* tmpl = a.grain_tmpl;
  const uint8_t* offs = a.grain_offs;
  uint16_t* frame = a.frame;
  const int bd = L.bit_depth;
  const int maxv = (1 << bd) - 1;
  const int lo = -(128 << (bd - 8)), hi = (256 << (bd - 8)) - 1 - (128 << (bd - 8));
  const int ntx = (L.out_w[0] + 63) / 64;
  const int tx0 = (t % ntx) * 64, ty0 = (t / ntx) * 32;
  const int cw = L.ss_x ? 44 : kLW, ch = L.ss_y ? 38 : kLH;
  const int chroma = g.cfl || g.num_cb > 0 || g.num_cr > 0;
  const uint16_t* luma = frame + L.plane_off[0];
  const int ls = L.stride[0];
  /* the three scaling tables in LDS (indexed by each sample's value) */
  for (int i = threadIdx.x; i < 768; i += 256) s_lut[i] = g.lut[i];
  __syncthreads();
  /* Each thread's samples (8 luma, up to 8 chroma per plane) go in three
   * batches: every load first (samples, luma, noise template), then the
   * arithmetic, then the stores, so no load waits behind another sample's
   * store. */
  constexpr int kPer = 64 * 32 / 256;
  for (int pl = 1; pl < 3 && chroma; ++pl) {
    if (!g.cfl && (pl == 1 ? g.num_cb : g.num_cr) <= 0) continue;
    NoiseCtx nc{tmpl + kLW * kLH + (pl - 1) * cw * ch, offs, cw, g.blocks, L.ss_x, L.ss_y, g.overlap, lo, hi};
    const int pw = L.out_w[pl], ph = L.out_h[pl];
    const int x0 = tx0 >> L.ss_x, y0 = ty0 >> L.ss_y;
    const int tw = 64 >> L.ss_x, th = 32 >> L.ss_y;
    const int* lut = s_lut + 256 * pl;
    const int mult = pl == 1 ? g.cb_mult : g.cr_mult;
    const int lmult = pl == 1 ? g.cb_luma_mult : g.cr_luma_mult;
    const int offset = pl == 1 ? g.cb_offset : g.cr_offset;
    uint16_t* plane = frame + L.plane_off[pl];
    const int st = L.stride[pl];
    const int lw = L.out_w[0];
    const int ltw = 6 - L.ss_x;
    int orig[kPer], avg[kPer], nv[kPer];
    bool ok[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = threadIdx.x + 256 * u;
      const int x = x0 + (i & (tw - 1)), y = y0 + (i >> ltw);
      ok[u] = i < tw * th && x < pw && y < ph;
      orig[u] = avg[u] = 0;
      if (ok[u]) {
        orig[u] = plane[(size_t)y * st + x];
        const int lx = x << L.ss_x, ly = y << L.ss_y;
        const int nx = lx + 1 < lw ? lx + 1 : lw - 1;
        const int l0 = luma[(size_t)ly * ls + lx];
        avg[u] = L.ss_x ? grnd(l0 + luma[(size_t)ly * ls + nx], 1) : l0;
      }
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = threadIdx.x + 256 * u;
      nv[u] = ok[u] ? nc.N(x0 + (i & (tw - 1)), y0 + (i >> ltw)) : 0;
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      if (!ok[u]) continue;
      const int i = threadIdx.x + 256 * u;
      const int x = x0 + (i & (tw - 1)), y = y0 + (i >> ltw);
      int index;
      if (g.cfl) {
        index = avg[u];
      } else {
        const int comb = avg[u] * (lmult - 128) + orig[u] * (mult - 128);
        index = clampi((comb >> 6) + (offset - 256) * (1 << (bd - 8)), 0, maxv);
      }
      const int gv = grnd(scale_lut(lut, index, bd) * nv[u], g.scaling_shift);
      plane[(size_t)y * st + x] = (uint16_t)clampi(orig[u] + gv, g.min_value, g.max_chroma);
    }
  }
  __syncthreads();
  if (g.num_y > 0) {
    NoiseCtx nc{tmpl, offs, kLW, g.blocks, 0, 0, g.overlap, lo, hi};
    uint16_t* plane = frame + L.plane_off[0];
    int orig[kPer], nv[kPer];
    bool ok[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = threadIdx.x + 256 * u;
      const int x = tx0 + (i & 63), y = ty0 + (i >> 6);
      ok[u] = x < L.out_w[0] && y < L.out_h[0];
      orig[u] = ok[u] ? plane[(size_t)y * ls + x] : 0;
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = threadIdx.x + 256 * u;
      nv[u] = ok[u] ? nc.N(tx0 + (i & 63), ty0 + (i >> 6)) : 0;
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      if (!ok[u]) continue;
      const int i = threadIdx.x + 256 * u;
      const int gv = grnd(scale_lut(s_lut, orig[u], bd) * nv[u], g.scaling_shift);
      plane[(size_t)(ty0 + (i >> 6)) * ls + tx0 + (i & 63)] = (uint16_t)clampi(orig[u] + gv, g.min_value, g.max_luma);
    }
  }
}

__global__ __launch_bounds__(256) void k_grain_apply(BatchDev B) {
  __shared__ int s_lut[768];
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKGrainApply);
  const int total = pre[B.njobs];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int j = find_job(pre, B.njobs, v);
    grain_tile(filter_args(B, j), v - pre[j], s_lut);
    __syncthreads();
  }
}

}  // namespace

int grain_tiles(const Layout& lay) { return (lay.out_w[0] + 63) / 64 * ((lay.out_h[0] + 31) / 32); }

hipError_t launch_grain_kernel(const BatchDev& b, int k, int total, int cap, hipStream_t s) {
  const dim3 grid(min(total, cap));
  switch (k) {
    case kKGrainTemplate: hipLaunchKernelGGL(k_grain_template, grid, dim3(64), 0, s, b); break;
    case kKGrainApply: hipLaunchKernelGGL(k_grain_apply, grid, dim3(256), 0, s, b); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace av1hip
