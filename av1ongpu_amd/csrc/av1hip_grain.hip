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

/* the noise of four neighbouring samples (of one noise block: x is a multiple
 * of 4), through whole words of the template */
struct NoiseCtx {
  const int16_t* t;   /* template of this plane, on a word */
  const uint8_t* offs;
  int tw, blocks, sx, sy, overlap, lo, hi;
  __device__ __forceinline__ void G(int s, int b, int i, int j, int* v) const {
    const int r = offs[s * blocks + b];
    const int ox = r >> 4, oy = r & 15;
    const int gx = sx ? 6 + ox : 9 + 2 * ox, gy = sy ? 6 + oy : 9 + 2 * oy;
    const int at = (gy + i) * tw + gx + j; /* rows are an even number of samples; 5 more stay in the row */
    const uint32_t* w = reinterpret_cast<const uint32_t*>(t + (at & ~1));
    const uint32_t w0 = w[0], w1 = w[1], w2 = w[2];
    const uint32_t p = __builtin_amdgcn_alignbit(w1, w0, at << 4), q = __builtin_amdgcn_alignbit(w2, w1, at << 4);
    v[0] = (int16_t)p;
    v[1] = (int)p >> 16;
    v[2] = (int16_t)q;
    v[3] = (int)q >> 16;
  }
  /* an overlap blend `k` samples from a block's or stripe's edge */
  __device__ __forceinline__ int blend(int sub, int k, int old, int v) const {
    return clampi(grnd(sub ? old * 23 + v * 22 : (k == 0 ? old * 27 + v * 17 : old * 17 + v * 27), 5), lo, hi);
  }
  /* the stripe buffer after the horizontal overlap blends */
  __device__ __forceinline__ void H(int s, int i, int x, int* v) const {
    const int lbw = 5 - sx, bw = 1 << lbw;
    const int b = x >> lbw, j = x & (bw - 1);
    G(s, b, i, j, v);
    if (overlap && b > 0 && j == 0) {
      int old[4];
      G(s, b - 1, i, bw, old);
      v[0] = blend(sx, 0, old[0], v[0]);
      if (!sx) v[1] = blend(0, 1, old[1], v[1]);
    }
  }
  /* the noise image after the vertical blends */
  __device__ __forceinline__ void N(int x, int y, int* v) const {
    const int lbh = 5 - sy, bh = 1 << lbh;
    const int s = y >> lbh, row = y & (bh - 1);
    H(s, row, x, v);
    if (overlap && s > 0 && row < (sy ? 1 : 2)) {
      int old[4];
      H(s - 1, row + bh, x, old);
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = blend(sy, row, old[k], v[k]);
    }
  }
};

/* a scaling table entry: its value and the step to the next one (0 from the
 * last one on, and at 8 bits nothing lies between two) */
__device__ __forceinline__ int scale_lut(const int2* lut, int index, int sh) {
  const int x = index >> sh;
  const int2 e = lut[x > 255 ? 255 : x];
  return e.x + grnd(e.y * (index - (x << sh)), sh);
}

__device__ __forceinline__ void unpack4(uint2 w, int* v) {
  v[0] = (int)(w.x & 0xffffu);
  v[1] = (int)(w.x >> 16);
  v[2] = (int)(w.y & 0xffffu);
  v[3] = (int)(w.y >> 16);
}

__device__ __forceinline__ void store4(uint16_t* dst, const int* v, int n) {
  if (n >= 4) {
    *reinterpret_cast<uint2*>(dst) =
        make_uint2((uint32_t)v[0] | (uint32_t)v[1] << 16, (uint32_t)v[2] | (uint32_t)v[3] << 16);
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (k < n) dst[k] = (uint16_t)v[k];
  }
}

/* 64x32 luma tiles (32x16 chroma at 4:2:0), 256 threads, four neighbouring
 * samples per lane and step: the loads, the template rows and the stores of a
 * step are one wide access each, and a noise block's offsets are looked up
 * once for the four. One sample per lane and step took 16.6 us on a 1080p
 * frame and 67 on a 2160p one; now 12 and 35 (over the 60 frames of the 1080p
 * clip 18.9 -> 13.5). */
__device__ void grain_tile(FArgs a, int t, int2* s_lut) {
  LayRef L = a.lay;
  const DevGrain& g = *a.plan.grain;
  const int16_t* tmpl = a.grain_tmpl;
  uint16_t* frame = a.frame;
  const int bd = L.bit_depth, sh = bd - 8;
  const int maxv = (1 << bd) - 1;
  const int lo = -(128 << sh), hi = (256 << sh) - 1 - (128 << sh);
  const int ntx = (L.out_w[0] + 63) / 64;
  const int tx0 = (t % ntx) * 64, ty0 = (t / ntx) * 32;
  const int cw = L.ss_x ? 44 : kLW, ch = L.ss_y ? 38 : kLH;
  const int chroma = g.cfl || g.num_cb > 0 || g.num_cr > 0;
  const uint16_t* luma = frame + L.plane_off[0];
  const int ls = L.stride[0], lw = L.out_w[0], lh = L.out_h[0];
  /* the three scaling tables in LDS (indexed by each sample's value) */
  for (int i = threadIdx.x; i < 768; i += 256) {
    const int v = g.lut[i];
    s_lut[i] = make_int2(v, (i & 255) < 255 ? g.lut[i + 1] - v : 0);
  }
  __syncthreads();
  const int quads = 512 >> (L.ss_x + L.ss_y), lq = 4 - L.ss_x; /* of a chroma plane; log2 of a row's */
  for (int e = threadIdx.x; chroma && e < 2 * quads; e += 256) {
    const int pl = __builtin_amdgcn_readfirstlane(e >= quads ? 2 : 1); /* quads is a multiple of a wave's */
    if (!g.cfl && (pl == 1 ? g.num_cb : g.num_cr) <= 0) continue;
    const int q = e - (pl - 1) * quads;
    const int x = (tx0 >> L.ss_x) + 4 * (q & ((1 << lq) - 1)), y = (ty0 >> L.ss_y) + (q >> lq);
    const int pw = L.out_w[pl], ph = L.out_h[pl];
    if (x >= pw || y >= ph) continue;
    const NoiseCtx nc{tmpl + kLW * kLH + (pl - 1) * cw * ch, a.grain_offs, cw, g.blocks, L.ss_x, L.ss_y, g.overlap, lo, hi};
    uint16_t* at = frame + L.plane_off[pl] + (size_t)y * L.stride[pl] + x;
    int orig[4], avg[4], nv[4], out[4];
    unpack4(*reinterpret_cast<const uint2*>(at), orig);
    const uint16_t* lr = luma + (size_t)(y << L.ss_y) * ls + (x << L.ss_x);
    if (L.ss_x) {
      const uint4 w = *reinterpret_cast<const uint4*>(lr);
      const uint32_t p[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int l0 = (int)(p[k] & 0xffffu);
        avg[k] = (l0 + (2 * (x + k) + 1 < lw ? (int)(p[k] >> 16) : l0) + 1) >> 1;
      }
    } else {
      unpack4(*reinterpret_cast<const uint2*>(lr), avg);
    }
    nc.N(x, y, nv);
    const int mult = (pl == 1 ? g.cb_mult : g.cr_mult) - 128;
    const int lmult = (pl == 1 ? g.cb_luma_mult : g.cr_luma_mult) - 128;
    const int offset = ((pl == 1 ? g.cb_offset : g.cr_offset) - 256) * (1 << sh);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      int index = avg[k];
      if (!g.cfl) index = clampi(((avg[k] * lmult + orig[k] * mult) >> 6) + offset, 0, maxv);
      out[k] = clampi(orig[k] + grnd(scale_lut(s_lut + 256 * pl, index, sh) * nv[k], g.scaling_shift), g.min_value,
                      g.max_chroma);
    }
    store4(at, out, pw - x);
  }
  /* chroma has read the tile's luma before the grain */
  __syncthreads();
  if (g.num_y <= 0) return;
  const NoiseCtx nc{tmpl, a.grain_offs, kLW, g.blocks, 0, 0, g.overlap, lo, hi};
  const int x = tx0 + 4 * ((int)threadIdx.x & 15);
  if (x >= lw) return;
  uint16_t* at[2];
  int y[2], nv[2][4];
  uint2 w[2] = {};
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    y[u] = ty0 + ((int)threadIdx.x >> 4) + 16 * u;
    at[u] = frame + L.plane_off[0] + (size_t)y[u] * ls + x;
    if (y[u] < lh) {
      w[u] = *reinterpret_cast<const uint2*>(at[u]);
      nc.N(x, y[u], nv[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (y[u] >= lh) continue;
    int orig[4], out[4];
    unpack4(w[u], orig);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      out[k] = clampi(orig[k] + grnd(scale_lut(s_lut, orig[k], sh) * nv[u][k], g.scaling_shift), g.min_value, g.max_luma);
    store4(at[u], out, lw - x);
  }
}

__global__ __launch_bounds__(256) void k_grain_apply(BatchDev B) {
  __shared__ int2 s_lut[768];
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
