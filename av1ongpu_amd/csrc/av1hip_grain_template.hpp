/*
 * Film grain templates (specification 7.18.3.2-3, the arithmetic of
 * av1gpu_kernels.h:3039-3122): white noise through the auto-regressive filter,
 * by single waves.
 *
 * A template is a chain: every sample needs its left neighbours and the row
 * above up to `lag` columns ahead. One wave runs a plane as a wavefront, lane
 * l on row l (then row l + 64), four columns behind the lane above, and every
 * sample a lane needs from the rows above streams through the lanes: its
 * windows of the three rows above shift by one column per step, the newest
 * values coming from the lane above by DPP, so a step is 14 two-tap products
 * from registers and one LDS write, 370 steps for luma. Before, a lane read its
 * 24 taps from LDS each step and three waves took 200 us for a frame's
 * templates, longer than the rest of a frame below 1080p; now two waves, each
 * building luma and then one chroma plane, take 104 us. (In the dependency
 * queue's launch instead of on a stream of its own it would save the two
 * crossings of hardware queues, about 20 us of a frame, where the queue lasts
 * longer than that, and lengthen it where it does not.)
 */
#ifndef AV1HIP_GRAIN_TEMPLATE_HPP
#define AV1HIP_GRAIN_TEMPLATE_HPP

#include "av1hip_internal.hpp"
#include "spec_tables.h"

namespace av1hip {
namespace grain {

constexpr int kLumaW = 82, kLumaH = 73;
constexpr int kGaussN = 2048;
/* LDS of a template wave: the luma template, the Gaussian sequence */
constexpr int kTemplateLds = (kLumaW * kLumaH + 4 + kGaussN) * 2;

constexpr unsigned lfsr_step(unsigned r) {
  return (r >> 1) | (((r ^ (r >> 1) ^ (r >> 3) ^ (r >> 12)) & 1u) << 15);
}
/* the LFSR `1 << k` template rows ahead, as 16x16 GF(2) matrices by columns */
struct Jump {
  uint16_t c[7][16];
};
constexpr Jump make_jump(int w) {
  Jump m{};
  for (int j = 0; j < 16; ++j) {
    unsigned v = 1u << j;
    for (int k = 0; k < w; ++k) v = lfsr_step(v);
    m.c[0][j] = (uint16_t)v;
  }
  for (int k = 1; k < 7; ++k)
    for (int j = 0; j < 16; ++j) {
      unsigned r = 0;
      for (int b = 0; b < 16; ++b)
        if (m.c[k - 1][j] & (1u << b)) r ^= m.c[k - 1][b];
      m.c[k][j] = (uint16_t)r;
    }
  return m;
}
__constant__ const Jump kJump82 = make_jump(82), kJump44 = make_jump(44);

/* the LFSR at the start of template row `row` */
__device__ __forceinline__ unsigned row_state(const Jump& m, unsigned seed, int row) {
  unsigned st = seed;
  for (int k = 0; k < 7; ++k) {
    unsigned r = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) r ^= (st >> j & 1u) ? m.c[k][j] : 0u;
    st = (row >> k) & 1 ? r : st;
  }
  return st;
}

__device__ __forceinline__ int clip(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }
/* the value of the lane above (lane 0: lane 63, whose row 63 it follows) */
__device__ __forceinline__ int from_above(int v) { return __builtin_amdgcn_mov_dpp(v, 0x13c, 0xf, 0xf, false); }

__device__ __forceinline__ uint32_t both(int lo, int hi) { return (uint32_t)(lo & 0xffff) | ((uint32_t)hi << 16); }
typedef short pair16 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int tap2(uint32_t v, uint32_t c, int acc) {
  return __builtin_amdgcn_sdot2(__builtin_bit_cast(pair16, v), __builtin_bit_cast(pair16, c), acc, false);
}

/* One plane by one wave, without a branch per lane. Windows hold pairs of
 * neighbouring 16-bit samples (columns k - 1, k in slot k % 7), so the taps
 * are 14 two-tap products. Luma finds its noise in `s_luma` and leaves the
 * template there. kChroma draws its noise (none: zeros) as it goes, a column
 * ahead, and reads the luma under the coming sample (av1gpu_kernels.h:
 * 3104-3112; `from_luma` false: no luma tap); the template goes to `out`. */
template <int kLag, bool kChroma>
__device__ __forceinline__ void plane(const AV1H_CMEM DevGrain& g, const AV1H_CMEM int* coeffs, int w, int h, bool noise,
                                      bool filter, unsigned seed, const Jump& jump, const int16_t* gauss,
                                      int16_t* s_luma, bool from_luma, int ss_x, int ss_y, int16_t* out) {
  const int lane = threadIdx.x & 63;
  const int bd = g.bit_depth;
  const int lo = -(128 << (bd - 8)), hi = (256 << (bd - 8)) - 1 - (128 << (bd - 8));
  /* 6 .. 9 and 0 .. 7 in a stream; below 1 nothing is shifted or rounded */
  const int shift = max(g.shift, 0), half = (1 << shift) >> 1;
  const int nshift = max(g.scale_shift, 0), nhalf = (1 << nshift) >> 1;
  /* pairs of coefficients: per row above (2 kLag + 1 columns) kLag pairs from
   * the right and the leftmost alone; of the own row's kLag likewise */
  constexpr int kCols = 2 * kLag + 1, kTaps = kCols * kLag + kLag;
  uint32_t ca[kLag > 0 ? kLag : 1][kLag + 1], co[2] = {0, 0};
#pragma unroll
  for (int r = 0; r < kLag; ++r) { /* r 0: the row above */
    const AV1H_CMEM int* c = coeffs + (kLag - 1 - r) * kCols + kLag;
#pragma unroll
    for (int i = 0; i < kLag; ++i) ca[r][i] = both(c[kLag - 2 * i - 1], c[kLag - 2 * i]);
    ca[r][kLag] = both(c[-kLag], 0);
  }
  if (kLag > 0) {
    const AV1H_CMEM int* c = coeffs + kCols * kLag + kLag;
    co[0] = both(kLag > 1 ? c[-2] : 0, c[-1]);
    co[1] = kLag > 2 ? both(c[-3], 0) : 0;
  }
  const int luma_coeff = kChroma && from_luma ? coeffs[kTaps] : 0;
  unsigned st = 0, st2 = 0;
  if (kChroma) {
    st = row_state(jump, seed, lane);
    st2 = h > 64 ? row_state(jump, seed, lane + 64) : 0;
  }
  uint32_t a1[7] = {}, a2[7] = {}, a3[7] = {}, own[7] = {};
  /* the coming column and its row; columns the filter reaches (none in the
   * first three rows) */
  constexpr int kNowhere = -(1 << 20);
  const int reach2 = filter ? w - 6 : 0;
  int x = lane < h ? -4 * lane - 1 : kNowhere, row = lane, reach = lane >= 3 ? reach2 : 0;
  int idx = row * w + x; /* of the coming column in the plane */
  int next = 0, l0 = 0, l1 = 0, l2 = 0, l3 = 0;
  bool next_in = false;
  const int steps = w + 4 * (h - 1) + 1;
  for (int s0 = 0; s0 < steps; s0 += 7) {
#pragma unroll
    for (int ph = 0; ph < 7; ++ph) {
      /* this column: its noise and luma were fetched a step ago */
      const int at = idx;
      const bool ar = (unsigned)(x - 3) < (unsigned)reach, in = (unsigned)x < (unsigned)w;
      const int nz = kChroma ? (next_in && noise ? (next + nhalf) >> nshift : 0) : next;
      const int lum = kChroma ? (l0 + l1 + l2 + l3 + ((1 << (ss_x + ss_y)) >> 1)) >> (ss_x + ss_y) : 0;
      ++x;
      ++idx;
      if (h > 64) { /* lane l goes on with row l + 64 (past the last: nowhere) */
        const bool wrap = x == 256;
        x = wrap ? (lane + 64 < h ? 0 : kNowhere) : x;
        idx = wrap ? (lane + 64) * w : idx;
        if (kChroma) row = wrap ? row + 64 : row;
        reach = wrap ? reach2 : reach;
        if (kChroma) st = wrap ? st2 : st;
      }
      if (kChroma) {
        next_in = (unsigned)x < (unsigned)w;
        const unsigned drawn = lfsr_step(st);
        st = next_in ? drawn : st;
        next = gauss[(st >> 5) & 2047];
        if (from_luma) {
          /* clamped for the lanes outside the filter's reach only: the last
           * luma row or column is read where a plane isn't subsampled */
          const int lx = max(0, min(((x - 3) << ss_x) + 3, kLumaW - 1 - ss_x)),
                    ly = max(0, min(((row - 3) << ss_y) + 3, kLumaH - 1 - ss_y));
          const int16_t* q = s_luma + ly * kLumaW + lx;
          l0 = q[0];
          if (ss_x) l1 = q[1];
          if (ss_y) {
            l2 = q[kLumaW];
            if (ss_x) l3 = q[kLumaW + 1];
          }
        }
      } else {
        next = s_luma[max(0, min(idx, w * h - 1))];
      }
      /* the rows above move on by one column, the newest sample in the high
       * half */
      const uint32_t n1 = (uint32_t)from_above((int)own[(ph + 6) % 7]), n2 = (uint32_t)from_above((int)a1[(ph + 3) % 7]),
                     n3 = (uint32_t)from_above((int)a2[(ph + 3) % 7]);
      a1[ph] = __builtin_amdgcn_perm(n1, a1[(ph + 6) % 7], 0x07060302u);
      a2[ph] = __builtin_amdgcn_perm(n2, a2[(ph + 6) % 7], 0x07060302u);
      a3[ph] = __builtin_amdgcn_perm(n3, a3[(ph + 6) % 7], 0x07060302u);
      int sum = half, sum2 = 0; /* two chains; the own row's taps last */
#pragma unroll
      for (int r = kLag - 1; r >= 0; --r) {
        const uint32_t(&v)[7] = r == 0 ? a1 : r == 1 ? a2 : a3;
#pragma unroll
        for (int i = 0; i < kLag; ++i) sum = tap2(v[(ph + 4 + kLag - 2 * i) % 7], ca[r][i], sum);
        sum2 = tap2(v[(ph + 5 - kLag) % 7], ca[r][kLag], sum2);
      }
      if (kChroma) sum2 += __mul24(lum, luma_coeff);
      if (kLag > 2) sum2 = tap2(own[(ph + 5) % 7], co[1], sum2);
      if (kLag > 0) sum = tap2(own[(ph + 6) % 7], co[0], sum);
      const int f = clip(nz + ((sum + sum2) >> shift), lo, hi);
      const int v = ar ? f : nz;
      own[ph] = __builtin_amdgcn_alignbit((uint32_t)v, own[(ph + 6) % 7], 16);
      if (kChroma) {
        if (in) out[at] = (int16_t)v;
      } else {
        s_luma[in ? at : kLumaW * kLumaH] = (int16_t)v; /* one spare place */
      }
    }
  }
}

template <bool kChroma>
__device__ __forceinline__ void plane_lag(const AV1H_CMEM DevGrain& g, const AV1H_CMEM int* coeffs, int w, int h, bool noise,
                                          bool filter, unsigned seed, const Jump& jump, const int16_t* gauss,
                                          int16_t* s_luma, bool from_luma, int ss_x, int ss_y, int16_t* out) {
  switch (g.lag) {
    case 0: plane<0, kChroma>(g, coeffs, w, h, noise, filter, seed, jump, gauss, s_luma, from_luma, ss_x, ss_y, out); break;
    case 1: plane<1, kChroma>(g, coeffs, w, h, noise, filter, seed, jump, gauss, s_luma, from_luma, ss_x, ss_y, out); break;
    case 2: plane<2, kChroma>(g, coeffs, w, h, noise, filter, seed, jump, gauss, s_luma, from_luma, ss_x, ss_y, out); break;
    default: plane<3, kChroma>(g, coeffs, w, h, noise, filter, seed, jump, gauss, s_luma, from_luma, ss_x, ss_y, out); break;
  }
}

/* Half of a frame's templates by one wave: half 0 luma (stored) and cb, half 1
 * luma again (for itself), cr and the offset draw of every (stripe, block).
 * `tmpl` receives luma (82x73) then cb and cr (cw x ch each); `lds` holds
 * kTemplateLds bytes. */
__device__ __forceinline__ void template_half(FArgs a, int half, void* lds) {
  const AV1H_CMEM DevGrain& g = *cmem(a.plan.grain);
  const int lane = threadIdx.x & 63;
  int16_t* s_luma = static_cast<int16_t*>(lds);
  int16_t* s_gauss = s_luma + kLumaW * kLumaH + 2; /* 4-byte aligned: 82 x 73 is even */
  for (int i0 = lane; i0 < kGaussN; i0 += 64 * 8) {
    int v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = av1t_spec_table[AV1T_OFF_GAUSSIAN + i0 + 64 * u];
#pragma unroll
    for (int u = 0; u < 8; ++u) s_gauss[i0 + 64 * u] = (int16_t)v[u];
  }
  __syncthreads();
  const unsigned seed = (unsigned)g.seed;
  if (half == 1) {
    /* per stripe block offsets (av1gpu_kernels.h:3236-3247) */
    for (int s = lane; s < g.stripes; s += 64) {
      unsigned r = seed;
      r ^= (unsigned)(((s * 37 + 178) & 255) << 8);
      r ^= (unsigned)((s * 173 + 105) & 255);
      for (int b = 0; b < g.blocks; ++b) {
        r = lfsr_step(r);
        a.grain_offs[s * g.blocks + b] = (uint8_t)((r >> 8) & 255);
      }
    }
  }
  /* luma noise, a row per lane (av1gpu_kernels.h:3070-3079) */
  const int nshift = max(g.scale_shift, 0), nhalf = (1 << nshift) >> 1;
  for (int row = lane; row < kLumaH; row += 64) {
    unsigned st = row_state(kJump82, seed, row);
    int16_t* to = s_luma + row * kLumaW;
#pragma unroll 2
    for (int x0 = 0; x0 < kLumaW / 41; ++x0)
#pragma unroll
      for (int u = 0; u < 41; u += 1) {
        st = lfsr_step(st);
        to[x0 * 41 + u] = g.num_y > 0 ? (int16_t)((s_gauss[(st >> 5) & 2047] + nhalf) >> nshift) : (int16_t)0;
      }
  }
  __syncthreads();
  const int ss_x = a.lay.ss_x, ss_y = a.lay.ss_y, cw = ss_x ? 44 : kLumaW, ch = ss_y ? 38 : kLumaH;
  plane_lag<false>(g, g.ar_y, kLumaW, kLumaH, true, g.num_y > 0, seed, kJump82, s_gauss, s_luma, false, 0, 0, nullptr);
  __syncthreads();
  if (half == 0) {
    const uint32_t* from = reinterpret_cast<const uint32_t*>(s_luma);
    uint32_t* to = reinterpret_cast<uint32_t*>(a.grain_tmpl);
    for (int i = lane; i < kLumaW * kLumaH / 2; i += 64) to[i] = from[i];
  }
  if (!(g.cfl || g.num_cb > 0 || g.num_cr > 0)) return;
  const bool noise = g.cfl || (half ? g.num_cr : g.num_cb) > 0;
  plane_lag<true>(g, half ? g.ar_cr : g.ar_cb, cw, ch, noise, true, seed ^ (half ? 0x49d8u : 0xb524u),
                  ss_x ? kJump44 : kJump82, s_gauss, s_luma, g.num_y > 0, ss_x, ss_y,
                  a.grain_tmpl + kLumaW * kLumaH + half * cw * ch);
}

}  // namespace grain
}  // namespace av1hip

#endif
