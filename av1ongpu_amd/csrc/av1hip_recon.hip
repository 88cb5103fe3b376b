/*
 * Reconstruction kernels for gfx950: prediction + inverse transform + residual.
 *
 * Per frame, in stream order:
 *   k_mc     - motion compensation of every inter block, four neighbouring
 *              samples per lane, straight into the frame;
 *   k_itx    - every transform block, grouped by its larger side G: G lanes
 *              per transform. Inter residuals are added into the frame, intra
 *              residuals are kept in a residual plane;
 *   k_queue  - a persistent work queue over the intra blocks: waves take
 *              blocks in dependency-level order, poll the packed edge words
 *              (or per cell epoch flags) of the neighbours a block reads until
 *              they are final, predict the block, add its residual and publish
 *              its own edges and cells. This replaces the
 *              reference's host wavefront schedule (src/core/engine.cpp:
 *              695-926): the dependencies are the same cells that scheduler
 *              waits for, but they resolve on the device as soon as each
 *              neighbour is done instead of one global wave at a time.
 *
 * This is the reference CPU backend's stage order inside a wave (inter, intra,
 * transforms, residual add; src/backends/cpu/cpu_backend.cpp:213-328) with
 * the transforms of intra blocks hoisted out of the dependency chain: their
 * residual does not depend on the prediction. The arithmetic is the
 * reference's (kernels/av1gpu_kernels.h), cited per function.
 */
#define AV1T_TABLE_QUAL static __constant__ const
#include "av1hip_internal.hpp"
#include "av1hip_itx.hpp"
#include "scan_order.hpp"

namespace av1hip {
/* the diagonal scans (scan_order.hpp), in device memory */
__device__ const av1scan::DiagTables kScanTab = av1scan::make_diag();

namespace {

#define SPEC(off) (av1t_spec_table + (off))

constexpr int kWork = 2048;            /* int32 intra work area (edges, CFL)    */

/* global (not generic) pointers: their accesses need no wait for LDS */
#define AV1H_GLOBAL __attribute__((address_space(1)))
#define AV1H_LDS __attribute__((address_space(3)))

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }
__device__ __forceinline__ int rnd2(int v, int n) { return n <= 0 ? v : (v + (1 << (n - 1))) >> n; }
__device__ __forceinline__ int rnd2s(int v, int n) {
  if (n <= 0) return v;
  return v >= 0 ? (v + (1 << (n - 1))) >> n : -((-v + (1 << (n - 1))) >> n);
}
__device__ __forceinline__ int rnd2s_add(int v, int n) { return (v + (1 << (n - 1)) + (v < 0 ? -1 : 0)) >> n; }
__device__ __forceinline__ int ilog2(int v) { return 31 - __builtin_clz(v); }

/* Samples other waves wrote in this launch are exchanged at device scope:
 * the stores and loads go to the level every XCD sees (the queue publishes a
 * block's cells only after its stores completed), so no cache writeback or
 * invalidate is needed around the dependency flags. */
__device__ __forceinline__ int ld_dev(const uint16_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(uint16_t* p, uint16_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* one wave per workgroup: the workgroup barrier is the wave barrier */
__device__ __forceinline__ void wsync() { __syncthreads(); }

__device__ int wave_sum(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

/* n words of 16-bit pairs from any such value's address, one wide load */
template <int N>
struct __attribute__((packed, aligned(2))) PairWords {
  uint32_t v[N];
};
template <int N>
__device__ __forceinline__ void load_words(const AV1H_GLOBAL uint16_t* p, uint32_t* s) {
  const AV1H_GLOBAL PairWords<N>* q = (const AV1H_GLOBAL PairWords<N>*)p;
#pragma unroll
  for (int t = 0; t < N; ++t) s[t] = q->v[t];
}
/* ------------------------------------------------------------------------ */
/* inverse transforms                                                        */
/* ------------------------------------------------------------------------ */

/* where a transform's residual goes: added to the frame within the sample
 * range (inter blocks, whose prediction is there), or stored as it is */
struct ItxOut {
  AV1H_GLOBAL uint16_t* dst; /* the transform's first sample */
  int stride, lo, hi;
  bool add;
};

/* One line of a pass (av1gpu_kernels.h:869-904 the rows, 907-930 the
 * columns): pass 0 the row `l` of N = w coefficients in place in LDS, pass 1
 * the column `l` of N = h values out to the picture. Both passes run this one
 * copy of the N point transform: a launch's time on frames up to 1080p is that
 * of fetching its instructions once per compute unit, so the second pass
 * finds them in the instruction cache (with a copy per pass and class, 185 and
 * 77 KB of code in the two launches, now 61 and 24: 1080p inter frame 27 + 15
 * -> 14 + 11 us, 2160p 29 + 34 -> 16 + 26, eight streams 20 + 43 -> 12 + 30;
 * the 24-bit form alone gave 27 -> 24). The addresses run along with the
 * values (the compiler would hold one per value, 396 registers). */
template <int N>
__device__ __forceinline__ void itx_line(int pass, int* tmp, int l, int w, int h, int tx_type, int lossless,
                                         int row_shift, int bd, int rect, const ItxOut& out) {
  if (l >= (pass ? w : h)) return;
  /* a line holds min(N, 32) coefficients (AV1 codes none beyond 32; rows
   * from 32 on are zero after the row pass): the other inputs are constant
   * zeros, which folds the first stages of the 64-point transform */
  constexpr int kIn = N < 32 ? N : 32;
  const int st = w + 1, step = pass ? st : 1;
  AV1H_LDS int* p = (AV1H_LDS int*)tmp + (pass ? l : l * st);
  if (!pass && l >= 32) {
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = 0;
    return;
  }
  int t[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    t[i] = i < kIn ? *p : 0;
    p += step;
    /* one running address, not one per value */
    if (i < kIn) asm volatile("" : "+v"(p));
  }
  p = (AV1H_LDS int*)tmp + (pass ? l : l * st);
  const int r = pass ? max(bd + 6, 16) : bd + 8;
  if (!lossless && itx::all_small<kIn>(t, r)) {
    if (rect && !pass) {
#pragma unroll
      for (int i = 0; i < kIn; ++i) t[i] = (__mul24(t[i], 2896) + 2048) >> 12;
    }
    itx::tx1d<true>(t, pass ? itx::col_kind(tx_type) : itx::row_kind(tx_type), 0, 0);
  } else {
    if (rect && !pass) {
#pragma unroll
      for (int i = 0; i < kIn; ++i) t[i] = itx::r12((int64_t)t[i] * 2896);
    }
    if (lossless) {
      if constexpr (N == 4) itx::iwht(t, pass ? 0 : 2);
    } else {
      itx::tx1d<false>(t, pass ? itx::col_kind(tx_type) : itx::row_kind(tx_type), -(1 << (r - 1)), (1 << (r - 1)) - 1);
    }
  }
  const int shift = lossless ? 0 : (pass ? 4 : row_shift), half = shift > 0 ? 1 << (shift - 1) : 0;
#pragma unroll
  for (int i = 0; i < N; ++i) t[i] = shift > 0 ? (t[i] + half) >> shift : t[i];
  if (!pass) {
    const int cr = 1 << (max(bd + 6, 16) - 1);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = clampi(t[i], -cr, cr - 1);
    return;
  }
  const int ud = itx::flip_ud(tx_type), hop = ud ? -out.stride : out.stride;
  AV1H_GLOBAL uint16_t* d = out.dst + (itx::flip_lr(tx_type) ? w - 1 - l : l) + (ud ? (N - 1) * out.stride : 0);
  AV1H_GLOBAL uint16_t* from = d;
  /* up to 32 rows at a time: their current samples are all loaded before any
   * is stored, so the adds do not wait on one load after another */
  constexpr int kB = N < 32 ? N : 32;
#pragma unroll
  for (int i0 = 0; i0 < N; i0 += kB) {
    int cur[kB];
#pragma unroll
    for (int u = 0; u < kB; ++u) cur[u] = 0;
    if (out.add) {
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        cur[u] = *from;
        from += hop;
        asm volatile("" : "+v"(from));
      }
    }
#pragma unroll
    for (int u = 0; u < kB; ++u) {
      *d = (uint16_t)clampi(cur[u] + t[i0 + u], out.lo, out.hi);
      d += hop;
      asm volatile("" : "+v"(d));
    }
  }
}

/* the line of the size `l2` (log2 points), instantiated only up to the
 * launch's largest class G */
template <int G>
__device__ __forceinline__ void itx_line_n(int l2, int pass, int* tmp, int l, int w, int h, int tx_type, int lossless,
                                           int row_shift, int bd, int rect, const ItxOut& out) {
  switch (l2) {
    case 2: itx_line<4>(pass, tmp, l, w, h, tx_type, lossless, row_shift, bd, rect, out); break;
    case 3: if constexpr (G >= 8) itx_line<8>(pass, tmp, l, w, h, tx_type, lossless, row_shift, bd, rect, out); break;
    case 4: if constexpr (G >= 16) itx_line<16>(pass, tmp, l, w, h, tx_type, lossless, row_shift, bd, rect, out); break;
    case 5: if constexpr (G >= 32) itx_line<32>(pass, tmp, l, w, h, tx_type, lossless, row_shift, bd, rect, out); break;
    default: if constexpr (G >= 64) itx_line<64>(pass, tmp, l, w, h, tx_type, lossless, row_shift, bd, rect, out); break;
  }
}

/* The transform blocks of one class (larger side 1 << lg, at most G): 1 << lg
 * lanes per transform, 64 >> lg transforms per wave, coefficients staged in LDS
 * between the row and the column pass. The residual of an inter block is added
 * into the frame (its prediction is already there); that of an intra block goes
 * to `res`, where the dependency queue adds it after the prediction. The lanes
 * per transform are a variable so that the classes of a launch share the code
 * of each size. */
template <int G>
__device__ __forceinline__ void itx_group(RArgs a, const int32_t* list, int n, int wg, int lg, int* s_tmp) {
  const int lanes = 1 << lg;
  const int grp = threadIdx.x >> lg, l = threadIdx.x & (lanes - 1);
  const int idx = wg * (64 >> lg) + grp;
  const bool live = idx < n;
  const int ti = live ? list[idx] : 0;
  DevTx tx;
  if (live) {
    tx = a.plan.tx[ti];
  } else {
    tx.w = tx.h = 4;
    tx.flags = kTxRaw;
    tx.plane = 0;
    tx.x = tx.y = tx.coef = tx.tx_type = tx.row_shift = tx.eob = 0;
  }
  int* tmp = s_tmp + grp * lanes * (lanes + 1);
  const int w = tx.w, h = tx.h, lw = ilog2(w), lh = ilog2(h);
  const bool to_res = (tx.flags & kTxToResidual) != 0;
  ItxOut out;
  out.stride = plane_vals(a.lay.stride)[tx.plane];
  out.dst = (to_res ? (AV1H_GLOBAL uint16_t*)a.res : (AV1H_GLOBAL uint16_t*)a.frame) +
            plane_vals(a.lay.plane_off)[tx.plane] + (int64_t)tx.y * out.stride + tx.x;
  out.lo = to_res ? -32768 : 0;
  out.hi = to_res ? 32767 : a.maxv;
  out.add = !to_res;
  const bool coded = live && !(tx.flags & kTxRaw);
  if (live && !coded) {
    /* raw residual (av1gpu_kernels.h:933-937), eight samples per lane at a
     * time: residuals and current samples loaded before any store */
    const int n = w * h;
    for (int i0 = l; i0 < n; i0 += 8 * lanes) {
      int r[8], cur[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i = i0 + u * lanes;
        r[u] = i < n ? a.plan.residual[tx.coef + i] : 0;
        cur[u] = i < n && out.add ? (int)out.dst[(i >> lw) * out.stride + (i & (w - 1))] : 0;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i = i0 + u * lanes;
        if (i < n) out.dst[(i >> lw) * out.stride + (i & (w - 1))] = (uint16_t)clampi(cur[u] + r[u], out.lo, out.hi);
      }
    }
  }
  if (coded) {
    /* the coefficients, eight neighbours (of one row, or of two rows of
     * four) per lane and step */
    const int cs = min(w, 32), cr = min(h, 32);
    const int lcs = ilog2(cs), st = w + 1, n = cs * cr, second = cs == 4 ? st - 4 : 0;
    auto put = [&](int i0, const int* v) {
      int* p = tmp + (i0 >> lcs) * st + (i0 & (cs - 1));
#pragma unroll
      for (int u = 0; u < 8; ++u) p[u + (u >= 4 ? second : 0)] = v[u];
    };
    if (a.plan.levels) {
      /* dequantised here from the coded levels: raster position i holds
       * scan index si, coded when below the transform's count */
      const DevDq q = a.plan.dq[ti];
      const int cls = av1scan::tx_class(tx.tx_type), lcw = lcs - 2, lch = ilog2(cr) - 2;
      const int count = tx.eob < n ? tx.eob : n;
      const int16_t* lv = a.plan.levels + q.level_off;
      for (int i0 = 8 * l; i0 < n; i0 += 8 * lanes) {
        int si[8], v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) si[u] = av1scan::scan_index(kScanTab.iscan, cls, lcw, lch, i0 + u);
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = si[u] < count ? (int)lv[si[u]] : 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + u;
          if (v[u])
            v[u] = av1scan::dequant(v[u], i ? q.ac_step : q.dc_step, q.qm_off >= 0 ? (int)a.plan.qm[q.qm_off + i] : -1,
                                    q.denom_shift, a.lay.bit_depth);
        }
        put(i0, v);
      }
    } else if (a.plan.coef16) {
      /* every coefficient a lane stages is loaded before the first LDS write */
      constexpr int kSteps = G < 32 ? 2 : 4;
      const AV1H_GLOBAL uint16_t* src = (const AV1H_GLOBAL uint16_t*)a.plan.coef + tx.coef;
      uint32_t c[kSteps][4];
#pragma unroll
      for (int k = 0; k < kSteps; ++k)
        if (8 * (l + k * lanes) < n) load_words<4>(src + 8 * (l + k * lanes), c[k]);
#pragma unroll
      for (int k = 0; k < kSteps; ++k) {
        if (8 * (l + k * lanes) >= n) break;
        int v[8];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          v[2 * u] = (int)(int16_t)c[k][u];
          v[2 * u + 1] = (int)c[k][u] >> 16;
        }
        put(8 * (l + k * lanes), v);
      }
    } else {
      const int32_t* src = static_cast<const int32_t*>(a.plan.coef) + tx.coef;
      for (int i0 = 8 * l; i0 < n; i0 += 8 * lanes) {
        int v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = src[i0 + u];
        put(i0, v);
      }
    }
  }
  const int lossless = (tx.flags & kTxLossless) ? 1 : 0, rect = (lw - lh == 1 || lh - lw == 1) ? 1 : 0;
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    __syncthreads();
    if (coded)
      itx_line_n<G>(pass ? lh : lw, pass, tmp, l, w, h, tx.tx_type, lossless, tx.row_shift, a.lay.bit_depth, rect, out);
  }
}

/* The classes [C0, C1) of a set in one launch, the larger first: two
 * launches (4-16 and 32-64) so that the small transforms, most of them, run
 * with the registers and LDS they need rather than the 64-point ones'. */
template <int C0, int C1>
__device__ __forceinline__ void itx_body(RArgs a, const int32_t* offs, int b, int* s_tmp) {
  for (int c = C1 - 1; c >= C0; --c) {
    const int o0 = offs[c], n = offs[c + 1] - o0;
    const int per = 16 >> c;
    const int wgs = (n + per - 1) / per;
    if (b < wgs) {
      const int32_t* list = a.plan.itx_list + o0;
      itx_group<(4 << (C1 - 1))>(a, list, n, b, c + 2, s_tmp);
      return;
    }
    b -= wgs;
  }
}

/* Both sets of every frame, the inter blocks' first: the intra blocks'
 * residuals are independent of the prediction, and one launch of both is
 * hardly longer than one of either (itx_line). */
template <int C0, int C1>
__global__ __launch_bounds__(64) void k_itx(BatchDev B) {
  constexpr int kG = 4 << (C1 - 1);
  __shared__ int s_tmp[64 * (kG + 1)];
  const AV1H_CMEM int32_t* pre0 = kernel_prefix(B, C0 == 0 ? kKItxInter : kKItxInterL);
  const AV1H_CMEM int32_t* pre1 = kernel_prefix(B, C0 == 0 ? kKItxIntra : kKItxIntraL);
  const int inter = pre0[B.njobs], total = inter + pre1[B.njobs];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int set = v >= inter;
    const AV1H_CMEM int32_t* pre = set ? pre1 : pre0;
    const int u = set ? v - inter : v;
    const int j = find_job(pre, B.njobs, u);
    RArgs a = recon_args(B, j);
    itx_body<C0, C1>(a, a.plan.itx_offs + set * (kTxClasses + 1), u - pre[j], s_tmp);
    __syncthreads();
  }
}

/* ------------------------------------------------------------------------ */
/* inter prediction                                                          */
/* ------------------------------------------------------------------------ */

__device__ __forceinline__ int filt_row(int cls, int extent) {
  if (extent > 4) return cls;
  if (cls == 0 || cls == 2) return 4;
  if (cls == 1) return 5;
  return cls;
}

struct McPos {
  int scaled;
  int bx, by, sub_x, sub_y;
  int ix, iy, fx, fy;          /* unscaled: integer offset and phase      */
  int sx0, sy0, stx, sty;      /* scaled: start and step in 1/1024         */
  __device__ __forceinline__ void col(int x, int* c, int* f) const {
    if (!scaled) {
      *c = bx + x + ix;
      *f = fx;
    } else {
      const int p = sx0 + stx * x;
      *c = p >> 10;
      *f = (p & 1023) >> 6;
    }
  }
  __device__ __forceinline__ void row(int y, int* c, int* f) const {
    if (!scaled) {
      *c = by + y + iy;
      *f = fy;
    } else {
      const int p = sy0 + sty * y;
      *c = p >> 10;
      *f = (p & 1023) >> 6;
    }
  }
};

/* the position arithmetic of av1gpu_kernels.h:1761-1763 (unscaled) and
 * 1819-1840 (scaled, 7.11.3.3) */
__device__ McPos mc_pos(int bx, int by, int mvx, int mvy, int sub_x, int sub_y, int scx, int scy) {
  McPos p;
  p.bx = bx;
  p.by = by;
  p.sub_x = sub_x;
  p.sub_y = sub_y;
  p.scaled = !(scx == (1 << 14) && scy == (1 << 14));
  const int mx = mvx * 2, my = mvy * 2;
  p.ix = mx >> (4 + sub_x);
  p.fx = (mx >> sub_x) & 15;
  p.iy = my >> (4 + sub_y);
  p.fy = (my >> sub_y) & 15;
  const int ox = (bx << 4) + ((2 * mvx) >> sub_x) + 8;
  const int oy = (by << 4) + ((2 * mvy) >> sub_y) + 8;
  p.sx0 = rnd2s_add(ox * scx - (8 << 14), 8) + 32;
  p.sy0 = rnd2s_add(oy * scy - (8 << 14), 8) + 32;
  p.stx = rnd2s_add(scx, 4);
  p.sty = rnd2s_add(scy, 4);
  return p;
}

__device__ const uint16_t* ref_plane(RArgs a, int slot, int plane) {
  const uint16_t* base = slot >= 0 ? a.pool + (size_t)slot * a.slot_size : a.frame;
  return base + a.lay.plane_off[plane];
}

/* ------------------------------------------------------------------------ */
/* the remaining inter tools, one sample at a time (av1gpu_kernels.h:        */
/* 1880-2326): global warp, wedge and difference weighted masks, OBMC,       */
/* inter/intra, intra block copy. They are rare, so they are computed the    */
/* direct way; samples of the frame being decoded are read at device scope.  */
/* ------------------------------------------------------------------------ */

typedef short mc_s2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int dot2(uint32_t s, int taps, int acc) {
  return __builtin_amdgcn_sdot2(__builtin_bit_cast(mc_s2, s), __builtin_bit_cast(mc_s2, taps), acc, false);
}
/* 8 samples in four words by the 8 taps of a filter row */
__device__ __forceinline__ int dot8(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t s3, int4 f, int acc) {
  return dot2(s3, f.w, dot2(s2, f.z, dot2(s1, f.y, dot2(s0, f.x, acc))));
}
__device__ __forceinline__ uint32_t pack2(int lo, int hi) { return (uint32_t)(lo & 0xffff) | ((uint32_t)hi << 16); }

/* the 8 samples x - 3 .. x + 4 of row y, clamped to the reference's visible
 * area, as four words. kCur: the frame being decoded, whose samples other
 * waves of this launch write (device scope loads); a finished reference is
 * read in one wide load where no clamp moves a sample. */
template <bool kCur>
__device__ __forceinline__ void ref_row8(const uint16_t* p, int stride, int x, int y, int x1, int y1, uint32_t* s) {
  const AV1H_GLOBAL uint16_t* row = (const AV1H_GLOBAL uint16_t*)p + (int64_t)clampi(y, 0, y1) * stride;
  if (!kCur && x >= 3 && x + 4 <= x1) {
    load_words<4>(row + x - 3, s);
    return;
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const AV1H_GLOBAL uint16_t* lo = row + clampi(x - 3 + 2 * t, 0, x1);
    const AV1H_GLOBAL uint16_t* hi = row + clampi(x - 2 + 2 * t, 0, x1);
    s[t] = kCur ? pack2(ld_dev((const uint16_t*)lo), ld_dev((const uint16_t*)hi)) : pack2(*lo, *hi);
  }
}

/* one sample of one reference through the two stage filter, unscaled or
 * scaled (av1gpu_kernels.h:1756-1857), its eight rows' loads all in flight */
template <bool kCur>
__device__ __forceinline__ int mc_tap(const uint16_t* ref, int stride, int ref_w, int ref_h, int sub_x, int sub_y,
                                      int scx, int scy, int bx, int by, int ew, int eh, int mvx, int mvy, int filt,
                                      int filt_v, int x, int y, int compound, int bd) {
  const int round0 = bd >= 12 ? 5 : 3;
  int round1 = compound ? 7 : 11;
  if (bd >= 12 && !compound) round1 -= 2;
  const McPos P = mc_pos(bx, by, mvx, mvy, sub_x, sub_y, scx, scy);
  int cx, fx, cy, fy;
  P.col(x, &cx, &fx);
  P.row(y, &cy, &fy);
  const int* hk = SPEC(AV1T_OFF_SUBPEL) + (filt_row(filt, ew) * 16 + fx) * 8;
  const int* vk = SPEC(AV1T_OFF_SUBPEL) + (filt_row(filt_v, eh) * 16 + fy) * 8;
  uint32_t s[8][4];
#pragma unroll
  for (int r = 0; r < 8; ++r) ref_row8<kCur>(ref, stride, cx, cy - 3 + r, ref_w - 1, ref_h - 1, s[r]);
  const int4 f = make_int4(pack2(hk[0], hk[1]), pack2(hk[2], hk[3]), pack2(hk[4], hk[5]), pack2(hk[6], hk[7]));
  int acc = 0;
#pragma unroll
  for (int r = 0; r < 8; ++r) acc += __mul24(dot8(s[r][0], s[r][1], s[r][2], s[r][3], f, 1 << (round0 - 1)) >> round0, vk[r]);
  return (acc + (1 << (round1 - 1))) >> round1;
}

__device__ __forceinline__ int warp_offs(int v) { return clampi(((v + 512) >> 10) + 64, 0, 192); }

/* one sample of a warped reference (av1gpu_kernels.h:1919-1958) */
template <bool kCur>
__device__ __forceinline__ int warp_tap(int sub_x, int sub_y, int ref_w, int ref_h, const AV1H_CMEM int* wp,
                                        const AV1H_CMEM int* abcd, const uint16_t* ref, int stride, int bx, int by,
                                        int x, int y, int bd, int compound) {
  const int* wf = SPEC(AV1T_OFF_WARP);
  const int i1 = (y & 7) - 4, i2 = (x & 7) - 4;
  const int64_t srcx = (int64_t)((bx + (x >> 3) * 8 + 4) << sub_x);
  const int64_t srcy = (int64_t)((by + (y >> 3) * 8 + 4) << sub_y);
  const int64_t dstx = (int64_t)wp[2] * srcx + (int64_t)wp[3] * srcy + wp[0];
  const int64_t dsty = (int64_t)wp[4] * srcx + (int64_t)wp[5] * srcy + wp[1];
  const int64_t x4 = dstx >> sub_x, y4 = dsty >> sub_y;
  const int ix4 = (int)(x4 >> 16), sx4 = (int)(x4 & 0xffff);
  const int iy4 = (int)(y4 >> 16), sy4 = (int)(y4 & 0xffff);
  const int round0 = bd >= 12 ? 5 : 3;
  int round1 = compound ? 7 : 11;
  if (bd >= 12 && !compound) round1 -= 2;
  const int oy = warp_offs(sy4 + abcd[2] * i2 + abcd[3] * i1);
  uint32_t s[8][4];
#pragma unroll
  for (int k = 0; k < 8; ++k) ref_row8<kCur>(ref, stride, ix4 + i2, iy4 + i1 - 3 + k, ref_w - 1, ref_h - 1, s[k]);
  int acc = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int* w = wf + warp_offs(sx4 + abcd[0] * i2 + abcd[1] * (i1 - 3 + k)) * 8;
    const int4 f = make_int4(pack2(w[0], w[1]), pack2(w[2], w[3]), pack2(w[4], w[5]), pack2(w[6], w[7]));
    acc += __mul24(dot8(s[k][0], s[k][1], s[k][2], s[k][3], f, 1 << (round0 - 1)) >> round0, wf[oy * 8 + k]);
  }
  return (acc + (1 << (round1 - 1))) >> round1;
}

/* the wedge master masks (av1gpu_kernels.h:1968-2014) */
__constant__ const int kWedgeEven[8] = {1, 4, 11, 27, 46, 58, 62, 63};
__constant__ const int kWedgeOdd[8] = {1, 2, 6, 18, 37, 53, 60, 63};
__constant__ const int kWedgeVert[6] = {2, 7, 21, 43, 57, 62};

__device__ int wedge_1d(int which, int j) {
  if (which == 2) return j < 29 ? 0 : (j >= 35 ? 64 : kWedgeVert[j - 29]);
  if (j < 28) return 0;
  if (j >= 36) return 64;
  return which == 0 ? kWedgeEven[j - 28] : kWedgeOdd[j - 28];
}
__device__ int wedge_ob63(int i, int j) {
  const int shift = (i & 1) ? 15 - (i >> 1) : 16 - (i >> 1);
  return wedge_1d(i & 1, clampi(j - shift, 0, 63));
}
__device__ int wedge_master(int dir, int i, int j) {
  switch (dir) {
    case 0: return wedge_1d(2, i);
    case 1: return wedge_1d(2, j);
    case 2: return wedge_ob63(j, i);
    case 4: return 64 - wedge_ob63(i, 63 - j);
    case 5: return 64 - wedge_ob63(j, 63 - i);
    default: return wedge_ob63(i, j);
  }
}
__device__ int wedge_px(BlkRef b, int i, int k) {
  const int m = wedge_master(b.wedge_dir, clampi(b.wedge_yoff + i, 0, 63), clampi(b.wedge_xoff + k, 0, 63));
  return b.wedge_flip ? 64 - m : m;
}

/* av1gpu_kernels.h:2025-2029 */
__device__ __forceinline__ int diffwtd(int d, int sh, int sign) {
  d = (d + (1 << (sh - 1))) >> sh;
  d = clampi(38 + (d >> 4), 0, 64);
  return sign ? 64 - d : d;
}

/* av1gpu_kernels.h:2076-2100 */
__constant__ const int kObmcMask[62] = {45, 64,
                                        39, 50, 59, 64,
                                        36, 42, 48, 53, 57, 61, 64, 64,
                                        34, 37, 40, 43, 46, 49, 52, 54, 56, 58, 60, 61, 64, 64, 64, 64,
                                        33, 35, 36, 38, 40, 41, 43, 44, 45, 47, 48, 50, 51, 52, 53, 55,
                                        56, 57, 58, 59, 60, 60, 61, 62, 64, 64, 64, 64, 64, 64, 64, 64};
__device__ __forceinline__ int obmc_mask(int len, int i) {
  const int base = len == 2 ? 0 : (len == 4 ? 2 : (len == 8 ? 6 : (len == 16 ? 14 : 30)));
  return kObmcMask[base + i];
}

/* inter/intra edges and prediction (av1gpu_kernels.h:2120-2205) */
struct IiCtx {
  const uint16_t* p; /* the block's top left sample in the frame being decoded */
  int stride, x, y, w, h, max_x, max_y, have_left, have_above, bd;
  __device__ int above(int i) const {
    const int mid = 1 << (bd - 1);
    if (!have_above) return have_left ? ld_dev(p - 1) : mid - 1;
    if (x + i > max_x) i = max_x - x;
    return ld_dev(p - stride + i);
  }
  __device__ int left(int i) const {
    const int mid = 1 << (bd - 1);
    if (!have_left) return have_above ? ld_dev(p - stride) : mid + 1;
    if (y + i > max_y) i = max_y - y;
    return ld_dev(p + (ptrdiff_t)i * stride - 1);
  }
};

__device__ int ii_sample(const IiCtx& c, int mode, int xs, int ys) {
  if (mode == 1) return c.above(xs);
  if (mode == 2) return c.left(ys);
  const int* sw = SPEC(AV1T_OFF_SM_WEIGHTS);
  if (mode == 3) {
    const int wy = sw[c.h - 4 + ys], wx = sw[c.w - 4 + xs];
    return rnd2(wy * c.above(xs) + (256 - wy) * c.left(c.h - 1) + wx * c.left(ys) + (256 - wx) * c.above(c.w - 1), 9);
  }
  int sum = 0;
  if (c.have_above && c.have_left) {
    for (int k = 0; k < c.w; ++k) sum += c.above(k);
    for (int k = 0; k < c.h; ++k) sum += c.left(k);
    return (sum + ((c.w + c.h) >> 1)) / (c.w + c.h);
  }
  if (c.have_left) {
    for (int k = 0; k < c.h; ++k) sum += c.left(k);
    return (sum + (c.h >> 1)) >> ilog2(c.h);
  }
  if (c.have_above) {
    for (int k = 0; k < c.w; ++k) sum += c.above(k);
    return (sum + (c.w >> 1)) >> ilog2(c.w);
  }
  return 1 << (c.bd - 1);
}

__device__ int ii_mask(BlkRef b, int sub_x, int sub_y, int xs, int ys) {
  if (b.flags & kIIWedge) {
    const int ny = sub_y + 1, nx = sub_x + 1, n = nx * ny;
    int sum = 0;
    for (int i = 0; i < ny; ++i)
      for (int k = 0; k < nx; ++k) sum += wedge_px(b, (ys << sub_y) + i, (xs << sub_x) + k);
    return n == 1 ? sum : (n == 2 ? (sum + 1) >> 1 : (sum + 2) >> 2);
  }
  if (b.ii_mode == 0) return 32;
  const int scale = 128 / max(b.w, b.h);
  int k = 0;
  if (b.ii_mode == 1)
    k = ys * scale;
  else if (b.ii_mode == 2)
    k = xs * scale;
  else if (b.ii_mode == 3)
    k = min(xs, ys) * scale;
  return SPEC(AV1T_OFF_II_WEIGHTS)[min(k, 127)];
}

/* Sample (xs, ys) of a block using any inter tool (av1gpu_kernels.h:2207-2326).
 * References of slot -1 (intra block copy) are the frame being decoded. */
template <bool kCur>
__device__ __forceinline__ int inter_sample(RArgs a, BlkRef b, int xs, int ys) {
  LayRef L = a.lay;
  const int p = b.plane, bd = L.bit_depth;
  const int sub_x = p > 0 ? L.ss_x : 0, sub_y = p > 0 ? L.ss_y : 0;
  const int stride = L.stride[p];
  const int compound = b.compound != 0;
  int v[2] = {0, 0};
  for (int r = 0; r < (compound ? 2 : 1); ++r) {
    const uint16_t* base = ref_plane(a, b.slot[r], p);
    const int cmp = r ? 1 : compound;
    v[r] = (b.flags & (r ? kWarp1 : kWarp0))
               ? warp_tap<kCur>(sub_x, sub_y, b.ref_w, b.ref_h, b.warp_params[r], b.warp_abcd[r], base, stride,
                          b.x, b.y, xs, ys, bd, cmp)
               : mc_tap<kCur>(base, stride, b.ref_w, b.ref_h, sub_x, sub_y, b.scale_x, b.scale_y, b.x, b.y, b.w,
                        b.h, b.mv[r][0], b.mv[r][1], b.filt, b.filt_v, xs, ys, cmp, bd);
  }
  int out = v[0];
  if (compound) {
    const int round0 = bd >= 12 ? 5 : 3;
    const int post = 2 * 7 - (round0 + 7);
    if (b.mask_kind != 0) {
      const int sh = post + (bd - 8);
      const int ny = sub_y + 1, nx = sub_x + 1;
      int sum = 0, n = 0;
      for (int i = 0; i < ny; ++i)
        for (int k = 0; k < nx; ++k) {
          const int lx = (xs << sub_x) + k, ly = (ys << sub_y) + i;
          int m;
          if (b.mask_kind == 1) {
            m = wedge_px(b, ly, lx);
            if (b.mask_sign) m = 64 - m;
          } else if (p == 0) {
            m = diffwtd(abs(v[0] - v[1]), sh, b.mask_sign);
          } else {
            /* the luma difference at the co-located luma sample */
            int lv[2];
            for (int r = 0; r < 2; ++r) {
              const uint16_t* lb = ref_plane(a, b.slot[r], 0);
              lv[r] = (b.flags & (r ? kMaskWarp1 : kMaskWarp0))
                          ? warp_tap<kCur>(0, 0, L.out_w[0], L.out_h[0], b.warp_params[r], b.warp_abcd[r], lb,
                                     L.stride[0], b.x << L.ss_x, b.y << L.ss_y, lx, ly, bd, 1)
                          : mc_tap<kCur>(lb, L.stride[0], L.out_w[0], L.out_h[0], 0, 0, b.scale_x, b.scale_y,
                                   b.x << L.ss_x, b.y << L.ss_y, b.w << sub_x, b.h << sub_y, b.mv[r][0],
                                   b.mv[r][1], b.filt, b.filt_v, lx, ly, 1, bd);
            }
            m = diffwtd(abs(lv[0] - lv[1]), sh, b.mask_sign);
          }
          sum += m;
          ++n;
        }
      const int m = n == 1 ? sum : (n == 2 ? (sum + 1) >> 1 : (sum + 2) >> 2);
      out = (m * v[0] + (64 - m) * v[1] + (1 << (5 + post))) >> (6 + post);
    } else if (b.compound == AV1H_COMPOUND_AVERAGE) {
      out = (v[0] + v[1] + (1 << post)) >> (1 + post);
    } else {
      out = (b.w0 * v[0] + b.w1 * v[1] + (1 << (3 + post))) >> (4 + post);
    }
  }
  out = clampi(out, 0, a.maxv);
  if ((b.flags & (kInterIntra | kInterDone)) == kInterIntra) {
    IiCtx c;
    c.p = a.frame + L.plane_off[p] + (size_t)b.y * stride + b.x;
    c.stride = stride;
    c.x = b.x;
    c.y = b.y;
    c.w = b.w;
    c.h = b.h;
    c.max_x = L.grid_w[p] - 1;
    c.max_y = L.grid_h[p] - 1;
    c.have_left = (b.flags & kHaveLeft) != 0;
    c.have_above = (b.flags & kHaveAbove) != 0;
    c.bd = bd;
    const int m = ii_mask(b, sub_x, sub_y, xs, ys);
    out = (m * ii_sample(c, b.ii_mode, xs, ys) + (64 - m) * out + 32) >> 6;
  }
  for (int k = 0; k < b.obmc_count; ++k) {
    const DevObmc& o = a.plan.obmc[b.obmc_first + k];
    if (xs < o.rx || xs >= o.rx + o.w || ys < o.ry || ys >= o.ry + o.h) continue;
    const int cj = xs - o.rx, ci = ys - o.ry;
    const int m = o.pass == 0 ? obmc_mask(o.h, ci) : obmc_mask(o.w, cj);
    const uint16_t* base = ref_plane(a, o.slot, p);
    int pred = mc_tap<false>(base, stride, b.ref_w, b.ref_h, sub_x, sub_y, b.scale_x, b.scale_y, b.x + o.rx,
                      b.y + o.ry, o.w, o.h, o.mvx, o.mvy, o.filt, o.filt_v, cj, ci, 0, bd);
    pred = clampi(pred, 0, a.maxv);
    out = (m * out + (64 - m) * pred + 32) >> 6;
  }
  return out;
}

/* inter_sample as a call, for the queue: inlined there it takes the registers
 * of every block's path */
template <bool kCur>
__device__ __noinline__ int queue_inter(const AV1H_CMEM ReconArgs* args, const AV1H_CMEM DevBlock* block, int xs, int ys) {
  return inter_sample<kCur>(*(const AV1H_CMEM ReconArgs*)sreg((int64_t)args),
                            *(const AV1H_CMEM DevBlock*)sreg((int64_t)block), xs, ys);
}

/* ------------------------------------------------------------------------ */
/* intra prediction                                                          */
/* ------------------------------------------------------------------------ */

constexpr int kEdge = 160;   /* edge entries (w + h <= 128, upsampled small) */
constexpr int kEdgeOff = 8;

/* The tables intra prediction indexes per lane (smooth weights, edge
 * kernels, filter intra taps), staged in LDS by the queue kernel: one
 * contiguous range of the specification table. */
constexpr int kTabLo = AV1T_OFF_SM_WEIGHTS, kTabHi = AV1T_OFF_II_WEIGHTS;
static_assert(AV1T_OFF_EDGE_KERNEL > kTabLo && AV1T_OFF_FILTER_INTRA > kTabLo && AV1T_OFF_FILTER_INTRA < kTabHi,
              "staged table range");
#define TAB(off) (tab + ((off) - kTabLo))

/* The edge preparation of a directional block (av1gpu_kernels.h:1452-1481,
 * with the filter of 1157-1173 and the upsampling of 1177-1191), its
 * choices precomputed on the host (DevBlock::dir_a): the corner filter, the
 * 5 tap filter of each edge into fa / fl and the 2x upsampling into ga / gl,
 * out of place so that each step is one LDS pass. `above` / `left` hold
 * entries -1 (the corner) .. w + h - 1; *ea / *el get the edges to predict
 * from. */
constexpr int kPrep1 = 2 * (kEdge + 2 * kEdgeOff), kPrep2 = 4 * (kEdge + 2 * kEdgeOff);
static_assert(kPrep2 + 2 * (kEdge + 2 * kEdgeOff) <= kWork, "edge preparation area");

/* What a queued block's work after its dependency wait reads of its
 * descriptor and of the frame's layout, loaded before the wait. Read after
 * it, each field is a scalar load, and the addresses chain several of them
 * one after another (the plane's strides and offsets, then the address):
 * about 0.3 us of each block's work after its wait (2.13 -> 1.85 us on the
 * 1080p key frame) that now overlaps the wait. */
struct QBlk {
  int x, y, w, h, plane, kind, flags, mode, dir_a, dir_b;
  int stride, max_x, max_y, maxv, bd;
  uint32_t epoch;
  /* global (not generic) pointers: their stores need no wait for LDS */
  AV1H_GLOBAL uint16_t* dst;     /* sample (x, y) of the block's plane in the frame */
  AV1H_GLOBAL uint64_t* row_pub; /* its last row's packed edge words (kEdgeRow)     */
  AV1H_GLOBAL uint64_t* col_pub; /* its last column's packed edge words (kEdgeCol)  */
};

__device__ __forceinline__ QBlk queued_block(RArgs a, BlkRef b) {
  LayRef L = a.lay;
  QBlk q;
  q.x = b.x;
  q.y = b.y;
  q.w = b.w;
  q.h = b.h;
  q.plane = __builtin_amdgcn_readfirstlane(b.plane);
  q.kind = b.kind;
  q.flags = b.flags;
  q.mode = b.mode;
  q.dir_a = b.dir_a;
  q.dir_b = b.dir_b;
  const int p = q.plane, sh = L.cell_shift[p];
  q.stride = L.stride[p];
  q.max_x = L.grid_w[p] - 1;
  q.max_y = L.grid_h[p] - 1;
  q.maxv = a.maxv;
  q.bd = L.bit_depth;
  q.epoch = a.epoch;
  q.dst = (AV1H_GLOBAL uint16_t*)(a.frame + L.plane_off[p] + (int64_t)q.y * q.stride + q.x);
  q.row_pub = (AV1H_GLOBAL uint64_t*)(a.edges + L.edge_row_off[p] +
                                      (int64_t)(((q.y + q.h) >> sh) - 1) * L.edge_row_words[p] + (q.x >> 1));
  q.col_pub = (AV1H_GLOBAL uint64_t*)(a.edges + L.edge_col_off[p] +
                                      (int64_t)(((q.x + q.w) >> sh) - 1) * L.edge_col_words[p] + (q.y >> 1));
  /* every field computed here, in scalar registers, before the caller's
   * wait: the compiler would otherwise sink the loads to their uses */
  asm volatile(""
               : "+s"(q.x), "+s"(q.y), "+s"(q.w), "+s"(q.h), "+s"(q.plane), "+s"(q.kind), "+s"(q.flags),
                 "+s"(q.mode), "+s"(q.dir_a), "+s"(q.dir_b), "+s"(q.stride), "+s"(q.max_x), "+s"(q.max_y),
                 "+s"(q.maxv), "+s"(q.bd), "+s"(q.epoch), "+s"(q.dst), "+s"(q.row_pub), "+s"(q.col_pub));
  return q;
}

__device__ void prepare_edges(const QBlk& b, const int* above, const int* left, int* work, const int* tab, int maxv,
                              int max_x, int max_y, const int** ea, const int** el) {
  const int lane = threadIdx.x, w = b.w, h = b.h, n = w + h;
  const int da = b.dir_a, pa = da & 511;
  const int stra = (da >> kDirStrA) & 7, strl = (da >> kDirStrL) & 7;
  int corner = above[-1];
  if (da & kDirCorner) corner = rnd2(left[0] * 5 + above[-1] * 6 + above[0] * 5, 4);
  const int sza = stra ? min(w, max_x - b.x + 1) + (pa < 90 ? h : 0) + 1 : 0;
  const int szl = strl ? min(h, max_y - b.y + 1) + (pa > 180 ? w : 0) + 1 : 0;
  int* fa = work + kPrep1 + kEdgeOff;
  int* fl = fa + kEdge + 2 * kEdgeOff;
  const int* ka = TAB(AV1T_OFF_EDGE_KERNEL) + 5 * max(stra - 1, 0);
  const int* kl = TAB(AV1T_OFF_EDGE_KERNEL) + 5 * max(strl - 1, 0);
  /* entry k of the filtered edge: the filter over entries clamp(k + q - 2,
   * -1, sz - 2) for 0 <= k <= sz - 2, the entry itself elsewhere */
  for (int j = lane - 1; j < 2 * n + 1; j += 64) {
    const bool is_a = j < n;
    const int k = is_a ? j : j - n - 1;
    const int* src = is_a ? above : left;
    const int sz = is_a ? sza : szl;
    int v;
    if (k >= 0 && k <= sz - 2) {
      const int* kk = is_a ? ka : kl;
      int acc = 0;
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        const int m = clampi(k + q - 2, -1, sz - 2);
        acc += kk[q] * (m < 0 ? corner : src[m]);
      }
      v = (acc + 8) >> 4;
    } else {
      v = k < 0 ? corner : src[k];
    }
    (is_a ? fa : fl)[k] = v;
  }
  wsync();
  *ea = fa;
  *el = fl;
  const int ua = (da & kDirUpA) != 0, ul = (da & kDirUpL) != 0;
  if (!ua && !ul) return;
  /* upsampled entry k: -2 the first tap, odd k = 2i - 1 the 4 tap
   * interpolation, even k = 2i the sample, past 2m - 2 (up to w + h - 1)
   * the entry as it was */
  const int na = ua ? w + (pa < 90 ? h : 0) : 0, nl = ul ? h + (pa > 180 ? w : 0) : 0;
  int* ga = work + kPrep2 + kEdgeOff;
  int* gl = ga + kEdge + 2 * kEdgeOff;
  const int span = 2 * n + 1; /* entries -2 .. 2n - 2 (upsampling needs w + h <= 16) */
  for (int j = lane; j < 2 * span; j += 64) {
    const bool is_a = j < span;
    const int m = is_a ? na : nl;
    const int k = (is_a ? j : j - span) - 2;
    if (m == 0 || (k > 2 * m - 2 && k > n - 1)) continue;
    const int* f = is_a ? fa : fl;
    auto t = [&](int i) { return f[clampi(i - 2, -1, m - 1)]; };
    int v;
    if (k == -2) {
      v = t(0);
    } else if (k <= 2 * m - 2) {
      if (k & 1) {
        const int i = (k + 1) >> 1;
        v = clampi(rnd2(-t(i) + 9 * t(i + 1) + 9 * t(i + 2) - t(i + 3), 4), 0, maxv);
      } else {
        v = t((k >> 1) + 2);
      }
    } else {
      v = f[k];
    }
    (is_a ? ga : gl)[k] = v;
  }
  wsync();
  if (ua) *ea = ga;
  if (ul) *el = gl;
}

/* The whole intra prediction of one block into s_pred (av1gpu_kernels.h:
 * 1578-1677 with the edges of 1108-1151 and the directional preparation of
 * 1452-1481). */
/* Polls a packed word until it carries `epoch`, with kPollDepth loads in
 * flight spaced about a round trip / kPollDepth apart (loads return in
 * order), so a word that lands is seen that much sooner than by one load
 * at a time. */
constexpr int kPollDepth = 1;
__device__ __forceinline__ uint64_t ld_word(const uint64_t* q) {
  return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ uint64_t poll_word(const uint64_t* q, uint32_t epoch, int limit, uint32_t* error) {
  uint64_t v[kPollDepth];
#pragma unroll
  for (int k = 0; k < kPollDepth; ++k) {
    if (k) __builtin_amdgcn_s_sleep(8);
    v[k] = ld_word(q);
  }
  for (int iter = 0;; iter += kPollDepth) {
#pragma unroll
    for (int k = 0; k < kPollDepth; ++k) {
      if ((uint32_t)(v[k] >> 32) == epoch) return v[k];
      if (kPollDepth == 1) __builtin_amdgcn_s_sleep(1);
      v[k] = ld_word(q);
    }
    if (iter >= limit) {
      atomicOr(error, 1u);
      return 0;
    }
  }
}

/* The edges of a block flagged kPackedEdges: its above row (x .. ae), left
 * column (y .. le) and corner come from the packed words its queued
 * neighbours published, each 64-bit word two samples and the epoch of the
 * frame that wrote them, so the one load per word is both the dependency
 * wait and the read (no cell flag, no second round trip to the frame), and
 * where the neighbour is outside the queue, from the frame without a wait.
 * Entries past ae / le repeat the last sample: only modes that read no
 * further than their dependencies reach use them. */
__device__ void gather_packed(RArgs a, BlkRef b, int* above, int* left, int alast, int llast, int mid,
                              uint32_t* error) {
  LayRef L = a.lay;
  const int p = b.plane, sh = L.cell_shift[p];
  const int x = b.x, y = b.y, n = b.w + b.h;
  const int ha = (b.flags & kHaveAbove) != 0, hl = (b.flags & kHaveLeft) != 0;
  const int ae = min(b.dep_x1, alast) - x, le = min(b.dep_y1, llast) - y;
  const uint64_t* rowp = a.edges + L.edge_row_off[p] + (int64_t)((y >> sh) - 1) * L.edge_row_words[p];
  const uint64_t* colp = a.edges + L.edge_col_off[p] + (int64_t)((x >> sh) - 1) * L.edge_col_words[p];
  /* samples of blocks outside the queue: final before it started */
  const int stride = L.stride[p];
  const uint16_t* fr = a.frame + L.plane_off[p] + (int64_t)y * stride + x;
  const uint32_t ma = (uint32_t)b.edge_mask_a, ml = (uint32_t)b.edge_mask_l;
  /* sample i of the above row / left column (block relative) */
  auto above_at = [&](int i) -> int {
    if ((ma >> (i >> sh)) & 1) {
      const uint64_t v = poll_word(rowp + ((x + i) >> 1), a.epoch, a.spin_limit, error);
      return (int)((v >> (16 * (i & 1))) & 0xffff);
    }
    return fr[i - stride];
  };
  auto left_at = [&](int i) -> int {
    if ((ml >> (i >> sh)) & 1) {
      const uint64_t v = poll_word(colp + ((y + i) >> 1), a.epoch, a.spin_limit, error);
      return (int)((v >> (16 * (i & 1))) & 0xffff);
    }
    return fr[(int64_t)i * stride - 1];
  };
  /* one pass over the corner (e = 0), above[0 .. n) and left[0 .. n), the
   * entries past the last sample a side depends on repeating it */
  for (int e = threadIdx.x; e < 2 * n + 1; e += 64) {
    int v;
    if (e == 0) {
      if (ha && hl) {
        if (b.flags & kCornerFrame) {
          v = fr[-stride - 1];
        } else {
          const uint64_t wv = poll_word((b.flags & kCornerRow) ? rowp + (x >> 1) - 1 : colp + (y >> 1) - 1, a.epoch,
                                        a.spin_limit, error);
          v = (int)((wv >> 16) & 0xffff); /* sample x - 1 of the row, or y - 1 of the column */
        }
      } else {
        v = ha ? above_at(0) : (hl ? left_at(0) : mid);
      }
      above[-1] = v;
      left[-1] = v;
    } else if (e <= n) {
      v = ha ? above_at(min(e - 1, ae)) : (hl ? left_at(0) : mid - 1);
      above[e - 1] = v;
    } else {
      v = hl ? left_at(min(e - n - 1, le)) : (ha ? above_at(0) : mid + 1);
      left[e - n - 1] = v;
    }
  }
}

/* The dependency wait of a kPackedEdges intra block: its edges into the
 * intra work area (entries -1 .. w + h - 1 of above / left, as
 * predict_intra reads them). */
__device__ void gather_edges(RArgs a, BlkRef b, int* work, uint32_t* error) {
  const int p = b.plane, w = b.w, h = b.h;
  gather_packed(a, b, work + kEdgeOff, work + kEdgeOff + kEdge + 2 * kEdgeOff,
                min(a.lay.grid_w[p] - 1, b.x + ((b.flags & kHaveAR) ? 2 * w : w) - 1),
                min(a.lay.grid_h[p] - 1, b.y + ((b.flags & kHaveBL) ? 2 * h : h) - 1), 1 << (a.lay.bit_depth - 1),
                error);
  wsync();
}

/* A queued block's last row and column as packed words (gather_packed). */
__device__ void write_edges(const QBlk& b, const uint16_t* pred) {
  const int w = b.w, h = b.h;
  const int nr = (b.flags & kEdgeRow) ? w >> 1 : 0, nc = (b.flags & kEdgeCol) ? h >> 1 : 0;
  const uint64_t tag = (uint64_t)b.epoch << 32;
  AV1H_GLOBAL uint64_t* rowp = b.row_pub;
  AV1H_GLOBAL uint64_t* colp = b.col_pub;
  const uint16_t* last = pred + (h - 1) * w;
  for (int k = threadIdx.x; k < nr + nc; k += 64) {
    uint64_t v;
    AV1H_GLOBAL uint64_t* q;
    if (k < nr) {
      v = tag | last[2 * k] | ((uint64_t)last[2 * k + 1] << 16);
      q = rowp + k;
    } else {
      const int j = k - nr;
      v = tag | pred[2 * j * w + w - 1] | ((uint64_t)pred[(2 * j + 1) * w + w - 1] << 16);
      q = colp + j;
    }
    __hip_atomic_store(q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

/* Residual samples of a block read before its wait (they do not depend on
 * the neighbours): one transform covering the block, at most 256 samples,
 * sample lane + 64 k in v[k]. */
struct EarlyRes {
  bool on;
  int16_t v[4];
};

/* Writes prediction samples f(s), s = 0 .. n - 1, clamped, into pred; with
 * an early residual (one transform over at most 256 samples, sample
 * lane + 64 k in er.v[k]) the residual is added and clamped in the same
 * pass (av1gpu_kernels.h:933-937). */
template <class F>
__device__ __forceinline__ void emit(int n, uint16_t* pred, const EarlyRes& er, int maxv, F f) {
  if (er.on) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int s = threadIdx.x + 64 * k;
      if (s < n) pred[s] = (uint16_t)clampi(clampi(f(s), 0, maxv) + er.v[k], 0, maxv);
    }
  } else {
    for (int s = threadIdx.x; s < n; s += 64) pred[s] = (uint16_t)clampi(f(s), 0, maxv);
  }
}

/* Returns whether the early residual is already added. */
__device__ bool predict_intra(RArgs a, BlkRef desc, const QBlk& b, int* work, uint16_t* pred, const int* tab,
                              const EarlyRes& er, uint32_t* error) {
  const int lane = threadIdx.x;
  const int w = b.w, h = b.h, lw = ilog2(w);
  const int stride = b.stride;
  const int bd = b.bd, maxv = b.maxv;
  const uint16_t* src = (const uint16_t*)b.dst;
  if (b.flags & kPalette) {
    for (int s = lane; s < w * h; s += 64) {
      const int y = s >> lw, x = s & (w - 1);
      pred[s] = (uint16_t)desc.palette[a.plan.palette[desc.palette_off + y * desc.palette_stride + x]];
    }
    wsync();
    return false;
  }
  int* above = work + kEdgeOff;
  int* left = work + kEdgeOff + kEdge + 2 * kEdgeOff;
  int* tmp = work + 2 * (kEdge + 2 * kEdgeOff);
  const int have_left = (b.flags & kHaveLeft) != 0, have_above = (b.flags & kHaveAbove) != 0;
  const int mid = 1 << (bd - 1);
  const int max_x = b.max_x, max_y = b.max_y;
  const int n = w + h;
  if (!(b.flags & kPackedEdges)) { /* packed edges: gathered by the caller (gather_edges) */
    const int alast = min(max_x, b.x + ((b.flags & kHaveAR) ? 2 * w : w) - 1);
    const int llast = min(max_y, b.y + ((b.flags & kHaveBL) ? 2 * h : h) - 1);
    for (int i = lane; i < n; i += 64) {
      above[i] = have_above ? ld_dev(src - stride + (min(b.x + i, alast) - b.x))
                            : (have_left ? ld_dev(src - 1) : mid - 1);
      left[i] = have_left ? ld_dev(src + (ptrdiff_t)(min(b.y + i, llast) - b.y) * stride - 1)
                          : (have_above ? ld_dev(src - stride) : mid + 1);
    }
    if (lane == 0) {
      int c;
      if (have_above && have_left)
        c = ld_dev(src - stride - 1);
      else if (have_above)
        c = ld_dev(src - stride);
      else if (have_left)
        c = ld_dev(src - 1);
      else
        c = mid;
      above[-1] = c;
      left[-1] = c;
    }
  }
  wsync();
  const int mode = b.mode;
  /* DC of the edges that exist (av1gpu_kernels.h:1430-1447) */
  auto dc_value = [&]() {
    int s = 0;
    if (have_above)
      for (int k = lane; k < w; k += 64) s += above[k];
    if (have_left)
      for (int k = lane; k < h; k += 64) s += left[k];
    s = wave_sum(s);
    if (have_above && have_left) return (s + ((w + h) >> 1)) / (w + h);
    if (have_left) return (s + (h >> 1)) >> ilog2(h);
    if (have_above) return (s + (w >> 1)) >> ilog2(w);
    return 1 << (bd - 1);
  };
  if (mode == AV1H_PRED_CFL) {
    /* chroma from luma (av1gpu_kernels.h:1603-1644) */
    const int dc = dc_value();
    const int sx = a.lay.ss_x, sy = a.lay.ss_y;
    const int luma_w = (b.x + w) << sx, luma_h = (b.y + h) << sy;
    const int xlim = luma_w - (1 << sx), ylim = luma_h - (1 << sy);
    const uint16_t* luma = a.frame + a.lay.plane_off[0];
    const int ls = a.lay.stride[0];
    int part = 0;
    for (int s = lane; s < w * h; s += 64) {
      const int y = s >> lw, x = s & (w - 1);
      const int ly = min((b.y + y) << sy, ylim), lx = min((b.x + x) << sx, xlim);
      int t = 0;
      for (int dy = 0; dy <= sy; ++dy)
        for (int dx = 0; dx <= sx; ++dx) t += ld_dev(luma + (size_t)(ly + dy) * ls + lx + dx);
      const int v = t << (3 - sx - sy);
      tmp[s] = v;
      part += v;
    }
    const int sum = wave_sum(part);
    const int shift = ilog2(w) + ilog2(h);
    const int avg = (sum + (1 << (shift - 1))) >> shift;
    emit(w * h, pred, er, maxv, [&](int s) { return dc + rnd2s(desc.cfl_alpha * (tmp[s] - avg), 6); });
    wsync();
    return true;
  }
  if ((b.flags & kFilterIntra) && w >= 4 && h >= 2) {
    /* recursive filter intra (av1gpu_kernels.h:1392-1427), one anti-diagonal
     * of 4x2 sub-blocks at a time: a sub-block reads only the ones above, to
     * its left and above-left */
    const int w4 = w >> 2, h2 = h >> 1;
    const int* taps = TAB(AV1T_OFF_FILTER_INTRA) + 56 * desc.fi_mode;
    for (int d = 0; d < w4 + h2 - 1; ++d) {
      const int c_lo = max(0, d - (h2 - 1)), c_hi = min(d, w4 - 1);
      const int nsub = c_hi - c_lo + 1;
      for (int idx = lane; idx < nsub * 8; idx += 64) {
        const int c4 = c_lo + (idx >> 3), k = idx & 7, r2 = d - c4;
        int pv[7];
        for (int i = 0; i < 5; ++i) {
          if (r2 == 0)
            pv[i] = above[(c4 << 2) + i - 1];
          else if (c4 == 0 && i == 0)
            pv[i] = left[(r2 << 1) - 1];
          else
            pv[i] = pred[((r2 << 1) - 1) * w + (c4 << 2) + i - 1];
        }
        for (int i = 5; i < 7; ++i)
          pv[i] = c4 == 0 ? left[(r2 << 1) + i - 5] : (int)pred[((r2 << 1) + i - 5) * w + (c4 << 2) - 1];
        int acc = 0;
        for (int i = 0; i < 7; ++i) acc += taps[k * 7 + i] * pv[i];
        pred[((r2 << 1) + (k >> 2)) * w + (c4 << 2) + (k & 3)] = (uint16_t)clampi(rnd2(acc, 4), 0, maxv);
      }
      wsync();
    }
    return false;
  }
  if (mode >= 1 && mode <= 8) {
    const int da = b.dir_a, pa = da & 511;
    const int ua = (da & kDirUpA) ? 1 : 0, ul = (da & kDirUpL) ? 1 : 0;
    const int* ea = above;
    const int* el = left;
    if (da & kDirFilter) prepare_edges(b, above, left, work, tab, maxv, max_x, max_y, &ea, &el);
    /* av1gpu_kernels.h:1245-1313 */
    const int dx = b.dir_b & 0xffff, dy = (int)((uint32_t)b.dir_b >> 16);
    emit(w * h, pred, er, maxv, [&](int s) {
      const int i = s >> lw, c = s & (w - 1);
      int v;
      if (pa < 90) {
        const int maxb = (w + h - 1) << ua;
        const int idx = (i + 1) * dx;
        const int base = (idx >> (6 - ua)) + (c << ua);
        const int sh = ((idx << ua) >> 1) & 31;
        v = base < maxb ? rnd2(ea[base] * (32 - sh) + ea[base + 1] * sh, 5) : ea[maxb];
      } else if (pa > 90 && pa < 180) {
        int idx = (c << 6) - (i + 1) * dx;
        int base = idx >> (6 - ua);
        if (base >= -(1 << ua)) {
          const int sh = ((idx * (1 << ua)) >> 1) & 31;
          v = rnd2(ea[base] * (32 - sh) + ea[base + 1] * sh, 5);
        } else {
          idx = (i << 6) - (c + 1) * dy;
          base = idx >> (6 - ul);
          const int sh = ((idx * (1 << ul)) >> 1) & 31;
          v = rnd2(el[base] * (32 - sh) + el[base + 1] * sh, 5);
        }
      } else if (pa > 180) {
        const int idx = (c + 1) * dy;
        const int base = (idx >> (6 - ul)) + (i << ul);
        const int sh = ((idx << ul) >> 1) & 31;
        v = rnd2(el[base] * (32 - sh) + el[base + 1] * sh, 5);
      } else {
        v = pa == 90 ? ea[c] : el[i];
      }
      return v;
    });
    wsync();
    return true;
  }
  if (mode >= AV1H_PRED_SMOOTH && mode <= AV1H_PRED_SMOOTH_H) {
    /* av1gpu_kernels.h:1333-1353 */
    const int* sw = TAB(AV1T_OFF_SM_WEIGHTS);
    emit(w * h, pred, er, maxv, [&](int s) {
      const int y = s >> lw, x = s & (w - 1);
      int v;
      if (mode == AV1H_PRED_SMOOTH) {
        const int wy = sw[h - 4 + y], wx = sw[w - 4 + x];
        v = rnd2(wy * above[x] + (256 - wy) * left[h - 1] + wx * left[y] + (256 - wx) * above[w - 1], 9);
      } else if (mode == AV1H_PRED_SMOOTH_V) {
        const int wy = sw[h - 4 + y];
        v = rnd2(wy * above[x] + (256 - wy) * left[h - 1], 8);
      } else {
        const int wx = sw[w - 4 + x];
        v = rnd2(wx * left[y] + (256 - wx) * above[w - 1], 8);
      }
      return v;
    });
    wsync();
    return true;
  }
  if (mode == AV1H_PRED_PAETH) {
    /* av1gpu_kernels.h:1364-1382 */
    emit(w * h, pred, er, maxv, [&](int s) {
      const int y = s >> lw, x = s & (w - 1);
      const int base = above[x] + left[y] - above[-1];
      const int pl = abs(base - left[y]), pt = abs(base - above[x]), ptl = abs(base - above[-1]);
      return (pl <= pt && pl <= ptl) ? left[y] : (pt <= ptl ? above[x] : above[-1]);
    });
    wsync();
    return true;
  }
  const int dc = clampi(dc_value(), 0, maxv);
  emit(w * h, pred, er, maxv, [&](int) { return dc; });
  wsync();
  return true;
}

/* ------------------------------------------------------------------------ */
/* block driver                                                              */
/* ------------------------------------------------------------------------ */

__device__ void store_block(const QBlk& b, const uint16_t* pred) {
  const int lw = ilog2(b.w);
  const int stride = b.stride;
  AV1H_GLOBAL uint16_t* dst = b.dst;
  if (b.flags & kSkipMark) {
    /* no block of this launch reads these samples (its readers take the
     * packed edge words): ordinary stores, written back through the L2 at
     * the end of the launch like any kernel's */
    for (int s = threadIdx.x; s < b.w * b.h; s += 64) dst[(size_t)(s >> lw) * stride + (s & (b.w - 1))] = pred[s];
    return;
  }
  for (int s = threadIdx.x; s < b.w * b.h; s += 64)
    __hip_atomic_store(dst + (size_t)(s >> lw) * stride + (s & (b.w - 1)), pred[s], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int64_t cell_index(LayRef L, int p, int x, int y) {
  return L.cell_off[p] + (int64_t)(y >> L.cell_shift[p]) * L.cells_w[p] + (x >> L.cell_shift[p]);
}

/* the cells of a block, flagged with this frame's epoch */
__device__ void mark_cells(RArgs a, BlkRef b, bool atomic) {
  const int p = b.plane, sh = a.lay.cell_shift[p];
  const int cw = max(b.w >> sh, 1), ch = max(b.h >> sh, 1);
  for (int i = threadIdx.x; i < cw * ch; i += 64) {
    const int cx = (b.x >> sh) + i % cw, cy = (b.y >> sh) + i / cw;
    if (cx >= a.lay.cells_w[p] || cy >= a.lay.cells_h[p]) continue;
    uint32_t* c = a.cells + a.lay.cell_off[p] + (int64_t)cy * a.lay.cells_w[p] + cx;
    if (atomic)
      __hip_atomic_store(c, a.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      *c = a.epoch;
  }
}

/* Wait until every cell the block reads carries this frame's epoch: the left
 * column, the above row and the corner the reference scheduler waits for
 * (engine.cpp:811-875), and for chroma from luma the co-located luma cells
 * (engine.cpp:908-916). */
__device__ void wait_cells(RArgs a, BlkRef b, uint32_t* error) {
  LayRef L = a.lay;
  const int p = b.plane, sh = L.cell_shift[p], cell = 1 << sh;
  const int gw = L.grid_w[p], gh = L.grid_h[p];
  int nl = 0, na = 0, nc = 0, ncfl = 0;
  int ly0 = b.y & ~(cell - 1), ax0 = b.x & ~(cell - 1);
  if (b.x - 1 >= 0 && b.dep_y1 >= ly0) nl = (min(b.dep_y1, gh - 1) - ly0) / cell + 1;
  if (b.y - 1 >= 0 && b.dep_x1 >= ax0) na = (min(b.dep_x1, gw - 1) - ax0) / cell + 1;
  if (nl < 0) nl = 0;
  if (na < 0) na = 0;
  if (b.dep_corner && b.x > 0 && b.y > 0) nc = 1;
  int lx0 = 0, ly0l = 0, lcw = 0;
  if (b.mode == AV1H_PRED_CFL && p > 0) {
    const int s0 = L.cell_shift[0];
    lx0 = (b.x << L.ss_x) >> s0;
    ly0l = (b.y << L.ss_y) >> s0;
    const int lx1 = min(((b.x + b.w - 1) << L.ss_x), L.grid_w[0] - 1) >> s0;
    const int ly1 = min(((b.y + b.h - 1) << L.ss_y), L.grid_h[0] - 1) >> s0;
    lcw = lx1 - lx0 + 1;
    ncfl = lcw * (ly1 - ly0l + 1);
  }
  int nr = 0, rcw = 0;
  if (b.flags & kIntraBC) {
    /* intra block copy: every cell of the source rectangle */
    rcw = b.dep_rx1 - b.dep_rx0 + 1;
    nr = rcw * (b.dep_ry1 - b.dep_ry0 + 1);
    if (rcw <= 0 || nr < 0) nr = 0;
  }
  const int total = nl + na + nc + ncfl + nr;
  if (total == 0) return;
  for (int iter = 0;; ++iter) {
    int ok = 1;
    for (int i = threadIdx.x; i < total; i += 64) {
      int64_t idx;
      if (i < nl)
        idx = cell_index(L, p, b.x - 1, ly0 + i * cell);
      else if (i < nl + na)
        idx = cell_index(L, p, ax0 + (i - nl) * cell, b.y - 1);
      else if (i < nl + na + nc)
        idx = cell_index(L, p, b.x - 1, b.y - 1);
      else if (i < nl + na + nc + ncfl) {
        const int k = i - nl - na - nc;
        idx = L.cell_off[0] + (int64_t)(ly0l + k / lcw) * L.cells_w[0] + lx0 + k % lcw;
      } else {
        const int k = i - nl - na - nc - ncfl;
        idx = L.cell_off[p] + (int64_t)(b.dep_ry0 + k / rcw) * L.cells_w[p] + b.dep_rx0 + k % rcw;
      }
      if (__hip_atomic_load(a.cells + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != a.epoch) ok = 0;
    }
    if (__all(ok)) break;
    if (iter >= a.spin_limit) {
      if (threadIdx.x == 0) atomicOr(error, 1u);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  /* the neighbours' samples are read with device scope loads issued after
   * the flag loads returned */
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

/* A block of the queue: the prediction, then the residuals of its transforms, which
 * k_itx computed before the queue started (av1gpu_kernels.h:933-937 for the
 * add), into `pred`; the caller stores it. */


/* one transform covers the block */
__device__ __forceinline__ bool one_transform(RArgs a, BlkRef b) {
  if (b.tx_count != 1) return false;
  const AV1H_CMEM DevTx& tx = cmem(a.plan.tx)[b.tx_first];
  return tx.x == b.x && tx.y == b.y && tx.w == b.w && tx.h == b.h;
}

__device__ __forceinline__ EarlyRes early_residual(RArgs a, BlkRef b, bool one) {
  EarlyRes e;
  e.on = one && b.w * b.h <= 256;
  if (!e.on) return e;
  const int p = b.plane, stride = a.lay.stride[p], lw = ilog2(b.w);
  const int16_t* r = a.res + a.lay.plane_off[p] + (int64_t)b.y * stride + b.x;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int s = threadIdx.x + 64 * k;
    e.v[k] = s < b.w * b.h ? r[(int64_t)(s >> lw) * stride + (s & (b.w - 1))] : 0;
  }
  return e;
}

/* ---- small intra blocks ------------------------------------------------
 * The blocks the queue's critical path is made of (4x4 .. 8x8, 4x16, 16x4:
 * at most 64 samples and 41 edge entries, three quarters and more of a
 * frame's queued blocks), one sample and one edge entry per lane, without
 * LDS. What bounds them is the latency of one wave from its neighbours'
 * words to its own, so everything that does not depend on the edges'
 * values - which word each lane polls, which entries and weights its sample
 * is made of, where it is stored - is computed into registers before the
 * wait; after it a sample takes one or two rounds of ds_bpermute between
 * the entries' lanes and a few multiply-adds, and the packed words are
 * formed by a DPP from the neighbouring lane. Against the LDS passes of
 * predict_intra for every size: queue of a 1080p key frame 2097 -> 1034 us
 * (768 levels), of a 426x240 one 497 -> 225 us, of a 1080p inter frame
 * 119 -> 66 us. Larger blocks keep those passes: they hold several samples
 * per lane, and one of them stands for several levels of small ones. */
constexpr int kSmallSamples = 64, kSmallEdge = 20; /* w * h, w + h */

__device__ __forceinline__ bool small_block(const QBlk& q, BlkRef b, bool one) {
  return q.kind == kIntra && (q.flags & (kPackedEdges | kFilterIntra | kPalette)) == kPackedEdges &&
         q.mode <= AV1H_PRED_PAETH && q.w * q.h <= kSmallSamples && q.w + q.h <= kSmallEdge &&
         (one || b.tx_count == 0);
}

/* the value of lane `at` / 4 */
__device__ __forceinline__ int from_lane(int at, int v) { return __builtin_amdgcn_ds_bpermute(at, v); }
template <int kCtrl, int kRows = 0xf>
__device__ __forceinline__ int dpp(int v) {
  return __builtin_amdgcn_update_dpp(0, v, kCtrl, kRows, 0xf, false);
}
/* the sum over the wave, in every lane's scalar: four row steps, two
 * broadcasts between the rows */
__device__ __forceinline__ int wave_total(int v) {
  v += dpp<0x111>(v);
  v += dpp<0x112>(v);
  v += dpp<0x114>(v);
  v += dpp<0x118>(v);
  v += dpp<0x142, 0xa>(v);
  v += dpp<0x143, 0xc>(v);
  return __builtin_amdgcn_readlane(v, 63);
}

#define AV1H_KEEP(...) asm volatile("" : __VA_ARGS__)

__device__ __forceinline__ void queue_small(RArgs a, BlkRef b, const QBlk& q, bool has_res, const int* tab,
                                            uint32_t* error, uint64_t* ready, bool trace) {
  LayRef L = a.lay;
  const int lane = threadIdx.x;
  const int w = q.w, h = q.h, n = w + h, lw = ilog2(w);
  const int x = lane & (w - 1), y = lane >> lw; /* this lane's sample */
  const bool sample = lane < w * h;
  int res = 0;
  if (has_res && sample)
    res = ((const AV1H_GLOBAL int16_t*)a.res)[(q.dst - (AV1H_GLOBAL uint16_t*)a.frame) + (int64_t)y * q.stride + x];
  const int sh = L.cell_shift[q.plane], mid = 1 << (q.bd - 1), maxv = q.maxv;
  const bool ha = (q.flags & kHaveAbove) != 0, hl = (q.flags & kHaveLeft) != 0;
  /* this lane's edge entry: lane n the corner, n + 1 + k above[k], n - 1 - k
   * left[k]; where it comes from as gather_packed has it */
  const int d = lane - n;
  const bool entry = lane <= 2 * n;
  const bool use_a = d >= 0 ? ha : (!hl && ha);
  const bool use_l = d <= 0 ? (hl && !(d == 0 && ha)) : (!ha && hl);
  int val = mid + (d > 0 ? -1 : (d < 0 ? 1 : 0)), half = 0;
  bool pend = false;
  AV1H_GLOBAL uint64_t* word = (AV1H_GLOBAL uint64_t*)a.edges;
  {
    const int alast = min(q.max_x, q.x + ((q.flags & kHaveAR) ? 2 * w : w) - 1);
    const int llast = min(q.max_y, q.y + ((q.flags & kHaveBL) ? 2 * h : h) - 1);
    const int ae = min(b.dep_x1, alast) - q.x, le = min(b.dep_y1, llast) - q.y;
    AV1H_GLOBAL uint64_t* rowp = word + L.edge_row_off[q.plane] + (int64_t)((q.y >> sh) - 1) * L.edge_row_words[q.plane];
    AV1H_GLOBAL uint64_t* colp = word + L.edge_col_off[q.plane] + (int64_t)((q.x >> sh) - 1) * L.edge_col_words[q.plane];
    const uint32_t ma = (uint32_t)b.edge_mask_a, ml = (uint32_t)b.edge_mask_l;
    const AV1H_GLOBAL uint16_t* from = q.dst;
    bool load = false;
    if (entry) {
      if (d == 0 && ha && hl) {
        if (q.flags & kCornerFrame) {
          load = true;
          from = q.dst - q.stride - 1;
        } else {
          pend = true;
          half = 16;
          word = (q.flags & kCornerRow) ? rowp + (q.x >> 1) - 1 : colp + (q.y >> 1) - 1;
        }
      } else if (use_a) {
        const int i = d > 0 ? min(d - 1, ae) : 0;
        if ((ma >> (i >> sh)) & 1) {
          pend = true;
          half = 16 * (i & 1);
          word = rowp + ((q.x + i) >> 1);
        } else {
          load = true;
          from = q.dst + i - q.stride;
        }
      } else if (use_l) {
        const int i = d < 0 ? min(-d - 1, le) : 0;
        if ((ml >> (i >> sh)) & 1) {
          pend = true;
          half = 16 * (i & 1);
          word = colp + ((q.y + i) >> 1);
        } else {
          load = true;
          from = q.dst + (int64_t)i * q.stride - 1;
        }
      }
    }
    if (load) val = *from; /* blocks outside the queue: final before it */
  }
  /* what the sample is made of */
  const int mode = q.mode;
  const bool dir = mode >= 1 && mode <= 8, smooth = mode >= AV1H_PRED_SMOOTH && mode <= AV1H_PRED_SMOOTH_H;
  const bool filt = dir && (((q.dir_a >> kDirStrA) | (q.dir_a >> kDirStrL)) & 7) != 0;
  const bool ups = dir && (q.dir_a & (kDirUpA | kDirUpL)) != 0;
  int i0 = 0, i1 = 0, i2 = 0, i3 = 0;  /* entries (lane * 4)             */
  int c0 = 0, c1 = 0, c2 = 0, c3 = 0;  /* weights                        */
  int j0 = 0, j1 = 0, j2 = 0, j3 = 0;  /* edge filter: tap entries       */
  int k0 = 16, k1 = 0, k2 = 0;         /* its kernel: centre, +-1, +-2   */
  if (dir) {
    const int pa = q.dir_a & 511, dx = q.dir_b & 0xffff, dy = (int)((uint32_t)q.dir_b >> 16);
    const int ua = (q.dir_a & kDirUpA) ? 1 : 0, ul = (q.dir_a & kDirUpL) ? 1 : 0;
    int left = 0, base, fr, up = 0;
    if (pa < 90) {
      const int idx = (y + 1) * dx;
      base = (idx >> (6 - ua)) + (x << ua);
      fr = ((idx << ua) >> 1) & 31;
      up = ua;
      if (base >= (n - 1) << ua) {
        base = n - 1;
        fr = up = 0;
      }
    } else if (pa > 90 && pa < 180) {
      int idx = (x << 6) - (y + 1) * dx;
      base = idx >> (6 - ua);
      up = ua;
      if (base < -(1 << ua)) {
        left = 1;
        idx = (y << 6) - (x + 1) * dy;
        base = idx >> (6 - ul);
        up = ul;
      }
      fr = ((idx * (1 << up)) >> 1) & 31;
    } else if (pa > 180) {
      const int idx = (x + 1) * dy;
      left = 1;
      base = (idx >> (6 - ul)) + (y << ul);
      fr = ((idx << ul) >> 1) & 31;
      up = ul;
    } else {
      left = pa == 180;
      base = left ? y : x;
      fr = 0;
    }
    /* entry k of the side as a lane address */
    auto at = [&](int k) { return 4 * (left ? n - 1 - k : n + 1 + k); };
    /* an upsampled entry 2i - 1 interpolates entries i - 2 .. i + 1 of the
     * edge, 2i is its entry i; of the pair base, base + 1 the odd one is
     * interpolated */
    const int odd = base & 1, m = (left ? h + (pa > 180 ? w : 0) : w + (pa < 90 ? h : 0)) - 1;
    if (up) {
      const int t = ((base + odd) >> 1) - 1 - odd;
      i0 = at(clampi(t, -1, m));
      i1 = at(clampi(t + 1, -1, m));
      i2 = at(clampi(t + 2, -1, m));
      i3 = at(clampi(t + 3, -1, m));
    } else {
      i1 = at(clampi(base, -1, n - 1));
      i2 = at(clampi(base + 1, -1, n - 1));
    }
    c0 = 32 - fr;
    c1 = fr;
    c2 = up && odd;
    c3 = up && !odd;
    if (filt) {
      const int stra = (q.dir_a >> kDirStrA) & 7, strl = (q.dir_a >> kDirStrL) & 7;
      const bool el = d < 0;
      const int str = el ? strl : stra, k = el ? -d - 1 : d - 1;
      const int last = (el ? min(h, q.max_y - q.y + 1) + (pa > 180 ? w : 0) : min(w, q.max_x - q.x + 1) + (pa < 90 ? h : 0)) - 1;
      auto te = [&](int i) { return 4 * (el ? n - 1 - clampi(i, -1, last) : n + 1 + clampi(i, -1, last)); };
      if (str && k >= 0 && k <= last) {
        const int* kk = TAB(AV1T_OFF_EDGE_KERNEL) + 5 * (str - 1);
        k0 = kk[2];
        k1 = kk[1];
        k2 = kk[0];
        j0 = te(k - 2);
        j1 = te(k - 1);
        j2 = te(k + 1);
        j3 = te(k + 2);
      }
    }
  } else if (smooth) {
    const int* sw = TAB(AV1T_OFF_SM_WEIGHTS);
    const int wy = mode == AV1H_PRED_SMOOTH_H ? 0 : sw[h - 4 + y], wx = mode == AV1H_PRED_SMOOTH_V ? 0 : sw[w - 4 + x];
    i1 = 4 * (n + 1 + x);
    i2 = 4 * (n - 1 - y);
    c0 = wy;
    c1 = mode == AV1H_PRED_SMOOTH_H ? 0 : 256 - wy;
    c2 = wx;
    c3 = mode == AV1H_PRED_SMOOTH_V ? 0 : 256 - wx;
  } else if (mode == AV1H_PRED_PAETH) {
    i1 = 4 * (n + 1 + x);
    i2 = 4 * (n - 1 - y);
  } else {
    /* DC: the entries it sums */
    c0 = ((ha && d > 0 && d <= w) || (hl && d < 0 && -d <= h)) ? 1 : 0;
  }
  /* DC: (sum + cnt / 2) / cnt as a high product with ceil(2^32 / cnt): exact
   * for sums below 2^32 / cnt^2 (cnt 4 .. 20, at most 20 samples of 12 bits) */
  const int cnt = (ha ? w : 0) + (hl ? h : 0);
  const uint32_t recip = cnt == 12 ? 0x15555556u : cnt == 20 ? 0x0ccccccdu : cnt ? 1u << (32 - ilog2(cnt)) : 0;
  /* where the sample and the packed words go: the last row's words by its
   * even columns, the last column's by the even rows, never the same lane */
  AV1H_GLOBAL uint16_t* dst = q.dst + (int64_t)y * q.stride + x;
  const bool row = sample && (q.flags & kEdgeRow) && y == h - 1 && !(x & 1);
  const bool col = sample && (q.flags & kEdgeCol) && x == w - 1 && !(y & 1);
  AV1H_GLOBAL uint64_t* pub = row ? q.row_pub + (x >> 1) : q.col_pub + (y >> 1);
  AV1H_KEEP("+v"(val), "+v"(res), "+v"(half), "+v"(word), "+v"(dst), "+v"(pub), "+v"(i0), "+v"(i1), "+v"(i2), "+v"(i3), "+v"(c0),
            "+v"(c1), "+v"(c2), "+v"(c3), "+v"(j0), "+v"(j1), "+v"(j2), "+v"(j3), "+v"(k0), "+v"(k1), "+v"(k2));
  /* the wait: every lane polls its entry's word until it carries this
   * frame's epoch (poll_word) */
  for (int iter = 0;; ++iter) {
    if (pend) {
      const uint64_t v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((uint32_t)(v >> 32) == q.epoch) {
        val = (int)(((uint32_t)v >> half) & 0xffffu);
        pend = false;
      }
    }
    if (!__any(pend)) break;
    if (iter >= a.spin_limit) {
      if (lane == 0) atomicOr(error, 1u);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  if (trace) *ready = (uint64_t)wall_clock64();
  int v;
  if (dir) {
    int e = val;
    if (filt)
      e = (k0 * val + k1 * (from_lane(j1, val) + from_lane(j2, val)) + k2 * (from_lane(j0, val) + from_lane(j3, val)) + 8) >> 4;
    int t1 = from_lane(i1, e), t2 = from_lane(i2, e);
    if (ups) {
      const int t0 = from_lane(i0, e), t3 = from_lane(i3, e);
      const int mv = clampi((9 * (t1 + t2) - t0 - t3 + 8) >> 4, 0, maxv);
      if (c2) t1 = mv;
      if (c3) t2 = mv;
    }
    v = (t1 * c0 + t2 * c1 + 16) >> 5;
  } else if (smooth) {
    const int bl = __builtin_amdgcn_readlane(val, w), ar = __builtin_amdgcn_readlane(val, n + w);
    v = c0 * from_lane(i1, val) + c1 * bl + c2 * from_lane(i2, val) + c3 * ar;
    v = mode == AV1H_PRED_SMOOTH ? (v + 256) >> 9 : (v + 128) >> 8;
  } else if (mode == AV1H_PRED_PAETH) {
    const int tl = __builtin_amdgcn_readlane(val, n), t = from_lane(i1, val), l = from_lane(i2, val);
    const int pl = abs(t - tl), pt = abs(l - tl), ptl = abs(t + l - 2 * tl);
    v = (pl <= pt && pl <= ptl) ? l : (pt <= ptl ? t : tl);
  } else {
    const int sum = wave_total(c0 ? val : 0);
    v = cnt ? (int)__umulhi((uint32_t)(sum + (cnt >> 1)), recip) : mid;
  }
  v = clampi(clampi(v, 0, maxv) + res, 0, maxv);
  /* packed words: this sample and the next one of its row / column */
  const int right = dpp<0xb1>(v); /* lane ^ 1 */
  if (q.flags & (kEdgeRow | kEdgeCol)) {
    int next = right;
    if (q.flags & kEdgeCol) {
      const int below = w == 4 ? dpp<0x104>(v) : (w == 8 ? dpp<0x108>(v) : from_lane(4 * (lane + w), v));
      if (col) next = below;
    }
    if (row || col)
      __hip_atomic_store(pub, ((uint64_t)q.epoch << 32) | ((uint32_t)next << 16) | (uint32_t)v, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  if (sample && !(x & 1)) {
    const uint32_t two = ((uint32_t)right << 16) | (uint32_t)v;
    AV1H_GLOBAL uint32_t* to = (AV1H_GLOBAL uint32_t*)dst;
    if (q.flags & kSkipMark)
      *to = two;
    else
      __hip_atomic_store(to, two, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

/* ---- large intra blocks --------------------------------------------------
 * The packed-edge blocks beyond 64 samples (8x16 .. 64x64) with one
 * transform or none. A chain of them is bound by the time from a block's
 * edges to its own last row and column, not by its samples: those are
 * predicted first, one packed word per lane, and published before the rest
 * of the block, whose pairs of samples then go straight from registers to
 * the frame. The polled words (two entries each, at most three per lane) are
 * all in flight together; edges and filtered edges lie in LDS. No size here
 * upsamples its edges (that takes w + h <= 16). A 16x16 block's work after
 * its wait, to the end of its stores, 3.2 -> 1.7 us, a 32x32 block's 12 ->
 * 3.8 us; queue of a 1080p key frame 1034 -> 801 us, of a 426x240 one 225 ->
 * 191 us, of a 2160p inter frame 164 -> 129 us. */
__device__ __forceinline__ bool big_block(const QBlk& q, BlkRef b, bool one) {
  return q.kind == kIntra && (q.flags & (kPackedEdges | kFilterIntra | kPalette)) == kPackedEdges &&
         q.mode <= AV1H_PRED_PAETH && q.w * q.h > kSmallSamples && !(q.dir_a & (kDirUpA | kDirUpL)) &&
         (one || b.tx_count == 0);
}

enum BigKind { kBigDc, kBigV, kBigH, kBigZ1, kBigZ2, kBigZ3, kBigSmooth, kBigSmoothV, kBigSmoothH, kBigPaeth };

/* sample (x, y) of a block of kind K: ea / el the edges, m0 .. m2 what the
 * kind needs of them or of the block (DC's value, the far corners) */
template <int K>
__device__ __forceinline__ int big_sample(int x, int y, int w, int h, int dx, int dy, const int* ea, const int* el,
                                          const int* sw, int m0, int m1) {
  if (K == kBigDc) return m0;
  if (K == kBigV) return ea[x];
  if (K == kBigH) return el[y];
  if (K == kBigZ1) {
    /* entries past the last repeat it, and a blend of equals is the value */
    const int idx = (y + 1) * dx, base = (idx >> 6) + x, fr = (idx >> 1) & 31, last = w + h - 1;
    return rnd2(ea[min(base, last)] * (32 - fr) + ea[min(base + 1, last)] * fr, 5);
  }
  if (K == kBigZ2) {
    const int ia = (x << 6) - (y + 1) * dx, il = (y << 6) - (x + 1) * dy;
    const bool up = (ia >> 6) >= -1;
    const int idx = up ? ia : il, fr = (idx >> 1) & 31;
    const int* e = (up ? ea : el) + (idx >> 6);
    return rnd2(e[0] * (32 - fr) + e[1] * fr, 5);
  }
  if (K == kBigZ3) {
    const int idx = (x + 1) * dy, fr = (idx >> 1) & 31;
    const int* e = el + (idx >> 6) + y;
    return rnd2(e[0] * (32 - fr) + e[1] * fr, 5);
  }
  if (K == kBigSmooth) {
    const int wy = sw[h - 4 + y], wx = sw[w - 4 + x];
    return rnd2(wy * ea[x] + (256 - wy) * m0 + wx * el[y] + (256 - wx) * m1, 9);
  }
  if (K == kBigSmoothV) {
    const int wy = sw[h - 4 + y];
    return rnd2(wy * ea[x] + (256 - wy) * m0, 8);
  }
  if (K == kBigSmoothH) {
    const int wx = sw[w - 4 + x];
    return rnd2(wx * el[y] + (256 - wx) * m1, 8);
  }
  const int t = ea[x], l = el[y]; /* Paeth: m0 the corner */
  const int pl = abs(t - m0), pt = abs(l - m0), ptl = abs(t + l - 2 * m0);
  return (pl <= pt && pl <= ptl) ? l : (pt <= ptl ? t : m0);
}

/* What a lane keeps of the block across the wait: its packed word's samples
 * and their residuals, the first residual pairs of its share of the block. */
struct BigLane {
  AV1H_GLOBAL uint64_t* pub;
  int x0, y0, x1, y1, r0, r1;
  bool on;
};
constexpr int kBigStep = 4; /* pairs per lane and step */

template <int K>
__device__ __forceinline__ void big_emit(const QBlk& q, const BigLane& g, uint32_t (&r)[kBigStep], bool has_res,
                                         const AV1H_GLOBAL uint32_t* res, int dx, int dy, const int* ea, const int* el,
                                         const int* sw, int m0, int m1) {
  const int w = q.w, h = q.h, maxv = q.maxv, lane = threadIdx.x, lw = ilog2(w);
  auto at = [&](int x, int y, int rv) {
    const int v = big_sample<K>(x, y, w, h, dx, dy, ea, el, sw, m0, m1);
    return clampi(clampi(v, 0, maxv) + rv, 0, maxv);
  };
  if (g.on) {
    const uint32_t two = (uint32_t)at(g.x0, g.y0, g.r0) | ((uint32_t)at(g.x1, g.y1, g.r1) << 16);
    __hip_atomic_store(g.pub, ((uint64_t)q.epoch << 32) | two, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  /* every pair of the block, the next step's residuals loaded ahead */
  const int pairs = (w * h) >> 1, half = q.stride >> 1;
  AV1H_GLOBAL uint32_t* dst = (AV1H_GLOBAL uint32_t*)q.dst;
  for (int p0 = 0; p0 < pairs; p0 += 64 * kBigStep) {
    uint32_t rn[kBigStep];
#pragma unroll
    for (int k = 0; k < kBigStep; ++k) {
      const int s = 2 * (p0 + 64 * (kBigStep + k) + lane);
      rn[k] = has_res && s < 2 * pairs ? res[(int64_t)(s >> lw) * half + ((s & (w - 1)) >> 1)] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kBigStep; ++k) {
      const int s = 2 * (p0 + 64 * k + lane);
      if (s >= 2 * pairs) break;
      const int x = s & (w - 1), y = s >> lw;
      const uint32_t two = (uint32_t)at(x, y, (int)(int16_t)r[k]) | ((uint32_t)at(x + 1, y, (int)r[k] >> 16) << 16);
      AV1H_GLOBAL uint32_t* to = dst + (int64_t)y * half + (x >> 1);
      if (q.flags & kSkipMark)
        *to = two;
      else
        __hip_atomic_store(to, two, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int k = 0; k < kBigStep; ++k) r[k] = rn[k];
  }
}

__device__ __forceinline__ void queue_big(RArgs a, BlkRef b, const QBlk& q, bool has_res, int* work, const int* tab,
                                          uint32_t* error, uint64_t* ready, bool trace) {
  LayRef L = a.lay;
  const int lane = threadIdx.x;
  const int w = q.w, h = q.h, n = w + h, lw = ilog2(w);
  const int sh = L.cell_shift[q.plane], mid = 1 << (q.bd - 1), maxv = q.maxv;
  const bool ha = (q.flags & kHaveAbove) != 0, hl = (q.flags & kHaveLeft) != 0;
  int* above = work + kEdgeOff;
  int* left = above + kEdge + 2 * kEdgeOff;
  /* residuals: the lane's border samples, its first pairs of the block */
  const AV1H_GLOBAL int16_t* res = (const AV1H_GLOBAL int16_t*)a.res + (q.dst - (AV1H_GLOBAL uint16_t*)a.frame);
  const AV1H_GLOBAL uint32_t* res2 = (const AV1H_GLOBAL uint32_t*)res;
  const int half = q.stride >> 1;
  BigLane g;
  {
    const bool row = lane < (w >> 1);
    const int j = row ? lane : lane - (w >> 1);
    g.x0 = row ? 2 * j : w - 1;
    g.x1 = row ? 2 * j + 1 : w - 1;
    g.y0 = row ? h - 1 : 2 * j;
    g.y1 = row ? h - 1 : 2 * j + 1;
    g.pub = row ? q.row_pub + j : q.col_pub + j;
    g.on = row ? (q.flags & kEdgeRow) != 0 : (q.flags & kEdgeCol) != 0 && j < (h >> 1);
    g.r0 = has_res && g.on ? res[(int64_t)g.y0 * q.stride + g.x0] : 0;
    g.r1 = has_res && g.on ? res[(int64_t)g.y1 * q.stride + g.x1] : 0;
  }
  uint32_t r[kBigStep];
#pragma unroll
  for (int k = 0; k < kBigStep; ++k) {
    const int s = 2 * (64 * k + lane);
    r[k] = has_res && s < w * h ? res2[(int64_t)(s >> lw) * half + ((s & (w - 1)) >> 1)] : 0u;
  }
  /* the words of the edges, two entries each: above 0 .. n - 1, left
   * 0 .. n - 1, the corner; sources as gather_packed has them */
  constexpr int kSlots = 3;
  const int words = n + 1;
  AV1H_GLOBAL uint64_t* word[kSlots];
  int v0[kSlots], v1[kSlots], s0[kSlots], s1[kSlots];
  bool pend[kSlots];
  {
    const int alast = min(q.max_x, q.x + ((q.flags & kHaveAR) ? 2 * w : w) - 1);
    const int llast = min(q.max_y, q.y + ((q.flags & kHaveBL) ? 2 * h : h) - 1);
    const int ae = min(b.dep_x1, alast) - q.x, le = min(b.dep_y1, llast) - q.y;
    AV1H_GLOBAL uint64_t* base = (AV1H_GLOBAL uint64_t*)a.edges;
    AV1H_GLOBAL uint64_t* rowp = base + L.edge_row_off[q.plane] + (int64_t)((q.y >> sh) - 1) * L.edge_row_words[q.plane];
    AV1H_GLOBAL uint64_t* colp = base + L.edge_col_off[q.plane] + (int64_t)((q.x >> sh) - 1) * L.edge_col_words[q.plane];
    const uint32_t ma = (uint32_t)b.edge_mask_a, ml = (uint32_t)b.edge_mask_l;
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      const int e = lane + 64 * u, nw = n >> 1;
      const int d = e < nw ? 1 : (e < 2 * nw ? -1 : 0), j = d < 0 ? e - nw : e;
      word[u] = base;
      pend[u] = false;
      s0[u] = s1[u] = 0;
      v0[u] = v1[u] = mid + (d > 0 ? -1 : (d < 0 ? 1 : 0));
      if (e >= words) continue;
      const bool use_a = d >= 0 ? ha : (!hl && ha), use_l = d <= 0 ? (hl && !(d == 0 && ha)) : (!ha && hl);
      if (d == 0 && ha && hl) {
        if (q.flags & kCornerFrame) {
          v0[u] = q.dst[-q.stride - 1];
        } else {
          pend[u] = true;
          s0[u] = s1[u] = 16;
          word[u] = (q.flags & kCornerRow) ? rowp + (q.x >> 1) - 1 : colp + (q.y >> 1) - 1;
        }
      } else if (use_a) {
        const int i0 = d > 0 ? min(2 * j, ae) : 0, i1 = d > 0 ? min(2 * j + 1, ae) : 0;
        if ((ma >> (i0 >> sh)) & 1) {
          pend[u] = true;
          s0[u] = 16 * (i0 & 1);
          s1[u] = 16 * (i1 & 1);
          word[u] = rowp + ((q.x + i0) >> 1);
        } else {
          v0[u] = q.dst[i0 - q.stride];
          v1[u] = q.dst[i1 - q.stride];
        }
      } else if (use_l) {
        const int i0 = d < 0 ? min(2 * j, le) : 0, i1 = d < 0 ? min(2 * j + 1, le) : 0;
        if ((ml >> (i0 >> sh)) & 1) {
          pend[u] = true;
          s0[u] = 16 * (i0 & 1);
          s1[u] = 16 * (i1 & 1);
          word[u] = colp + ((q.y + i0) >> 1);
        } else {
          v0[u] = q.dst[(int64_t)i0 * q.stride - 1];
          v1[u] = q.dst[(int64_t)i1 * q.stride - 1];
        }
      }
    }
  }
#pragma unroll
  for (int u = 0; u < kSlots; ++u) AV1H_KEEP("+v"(word[u]), "+v"(v0[u]), "+v"(v1[u]), "+v"(s0[u]), "+v"(s1[u]));
  AV1H_KEEP("+v"(g.pub), "+v"(g.r0), "+v"(g.r1), "+v"(g.x0), "+v"(g.x1), "+v"(g.y0), "+v"(g.y1));
  for (int iter = 0;; ++iter) {
    uint64_t v[kSlots];
#pragma unroll
    for (int u = 0; u < kSlots; ++u)
      v[u] = pend[u] ? __hip_atomic_load(word[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    bool any = false;
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      if (pend[u] && (uint32_t)(v[u] >> 32) == q.epoch) {
        v0[u] = (int)(((uint32_t)v[u] >> s0[u]) & 0xffffu);
        v1[u] = (int)(((uint32_t)v[u] >> s1[u]) & 0xffffu);
        pend[u] = false;
      }
      any = any || pend[u];
    }
    if (!__any(any)) break;
    if (iter >= a.spin_limit) {
      if (lane == 0) atomicOr(error, 1u);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  if (trace) *ready = (uint64_t)wall_clock64();
#pragma unroll
  for (int u = 0; u < kSlots; ++u) {
    const int e = lane + 64 * u, nw = n >> 1;
    if (e >= words) continue;
    if (e < 2 * nw) {
      int* to = e < nw ? above + 2 * e : left + 2 * (e - nw);
      to[0] = v0[u];
      to[1] = v1[u];
    } else {
      above[-1] = left[-1] = v0[u];
    }
  }
  wsync();
  const int mode = q.mode, pa = q.dir_a & 511, dx = q.dir_b & 0xffff, dy = (int)((uint32_t)q.dir_b >> 16);
  const int* ea = above;
  const int* el = left;
  const int* sw = TAB(AV1T_OFF_SM_WEIGHTS);
  if (mode >= 1 && mode <= 8) {
    const int stra = (q.dir_a >> kDirStrA) & 7, strl = (q.dir_a >> kDirStrL) & 7;
    if ((q.dir_a & kDirCorner) || stra || strl) {
      /* the entries the zone reads (av1gpu_kernels.h:1157-1173): above of
       * w + h, left of w + h, or the w + h around the corner */
      int corner = above[-1];
      if (q.dir_a & kDirCorner) corner = rnd2(left[0] * 5 + above[-1] * 6 + above[0] * 5, 4);
      int* fa = work + kPrep1 + kEdgeOff;
      int* fl = fa + kEdge + 2 * kEdgeOff;
      const int na = pa < 90 ? n : (pa > 180 ? 0 : w);
      for (int e = lane; e <= n; e += 64) {
        const bool is_l = e > na;
        const int k = is_l ? e - na - 1 : e - 1; /* -1: the corner */
        const int* src = is_l ? left : above;
        const int str = is_l ? strl : stra;
        const int last = is_l ? min(h, q.max_y - q.y + 1) + (pa > 180 ? w : 0) - 1 : min(w, q.max_x - q.x + 1) + (pa < 90 ? h : 0) - 1;
        int v = k < 0 ? corner : src[k];
        if (str && k >= 0 && k <= last) {
          const int* kk = TAB(AV1T_OFF_EDGE_KERNEL) + 5 * (str - 1);
          int acc = 8;
#pragma unroll
          for (int t = 0; t < 5; ++t) {
            const int m = clampi(k + t - 2, -1, last);
            acc += kk[t] * (m < 0 ? corner : src[m]);
          }
          v = acc >> 4;
        }
        if (k < 0)
          fa[-1] = fl[-1] = v;
        else
          (is_l ? fl : fa)[k] = v;
      }
      wsync();
      ea = fa;
      el = fl;
    }
    if (pa == 90)
      big_emit<kBigV>(q, g, r, has_res, res2, dx, dy, ea, el, sw, 0, 0);
    else if (pa == 180)
      big_emit<kBigH>(q, g, r, has_res, res2, dx, dy, ea, el, sw, 0, 0);
    else if (pa < 90)
      big_emit<kBigZ1>(q, g, r, has_res, res2, dx, dy, ea, el, sw, 0, 0);
    else if (pa < 180)
      big_emit<kBigZ2>(q, g, r, has_res, res2, dx, dy, ea, el, sw, 0, 0);
    else
      big_emit<kBigZ3>(q, g, r, has_res, res2, dx, dy, ea, el, sw, 0, 0);
  } else if (mode == AV1H_PRED_SMOOTH) {
    big_emit<kBigSmooth>(q, g, r, has_res, res2, dx, dy, ea, el, sw, left[h - 1], above[w - 1]);
  } else if (mode == AV1H_PRED_SMOOTH_V) {
    big_emit<kBigSmoothV>(q, g, r, has_res, res2, dx, dy, ea, el, sw, left[h - 1], 0);
  } else if (mode == AV1H_PRED_SMOOTH_H) {
    big_emit<kBigSmoothH>(q, g, r, has_res, res2, dx, dy, ea, el, sw, 0, above[w - 1]);
  } else if (mode == AV1H_PRED_PAETH) {
    big_emit<kBigPaeth>(q, g, r, has_res, res2, dx, dy, ea, el, sw, above[-1], 0);
  } else {
    /* DC (av1gpu_kernels.h:1430-1447): w + h <= 128 samples, two per lane */
    int s = 0;
    if (ha && lane < w) s += above[lane];
    if (hl && lane < h) s += left[lane];
    s = wave_total(s);
    int dc = mid;
    if (ha && hl)
      dc = (s + (n >> 1)) / n;
    else if (hl)
      dc = (s + (h >> 1)) >> ilog2(h);
    else if (ha)
      dc = (s + (w >> 1)) >> lw;
    big_emit<kBigDc>(q, g, r, has_res, res2, dx, dy, ea, el, sw, clampi(dc, 0, maxv), 0);
  }
}

/* ---- inter/intra blocks whose inter half is done -----------------------
 * Before the wait the inter samples go to `pred` and the blend masks to bytes
 * in the work area; after it the edges are read once (the per sample path
 * read each DC sample's w + h neighbours again), then every sample is a blend
 * of values in LDS (av1gpu_kernels.h:2120-2205). */
constexpr int kIiMask = 512; /* the masks' place in the work area, in words */
static_assert(kIiMask + 64 * 64 / 4 <= kWork, "inter/intra masks");

__device__ __forceinline__ void ii_ahead(RArgs a, BlkRef b, const QBlk& q, int* work, uint16_t* pred) {
  const int n = q.w * q.h, lw = ilog2(q.w);
  const int sub_x = q.plane > 0 ? a.lay.ss_x : 0, sub_y = q.plane > 0 ? a.lay.ss_y : 0;
  uint8_t* mask = reinterpret_cast<uint8_t*>(work + kIiMask);
  for (int s0 = threadIdx.x; s0 < n; s0 += 64 * 4) {
    uint16_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = s0 + 64 * u;
      v[u] = s < n ? q.dst[(int64_t)(s >> lw) * q.stride + (s & (q.w - 1))] : 0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = s0 + 64 * u;
      if (s >= n) break;
      pred[s] = v[u];
      mask[s] = (uint8_t)ii_mask(b, sub_x, sub_y, s & (q.w - 1), s >> lw);
    }
  }
}

__device__ __forceinline__ void ii_blend(BlkRef b, const QBlk& q, int* work, uint16_t* pred) {
  const int lane = threadIdx.x, w = q.w, h = q.h, lw = ilog2(w), mode = b.ii_mode;
  const bool ha = (q.flags & kHaveAbove) != 0, hl = (q.flags & kHaveLeft) != 0;
  int* above = work;
  int* left = work + 64;
  const uint8_t* mask = reinterpret_cast<const uint8_t*>(work + kIiMask);
  IiCtx c;
  c.p = (const uint16_t*)q.dst;
  c.stride = q.stride;
  c.x = q.x;
  c.y = q.y;
  c.w = w;
  c.h = h;
  c.max_x = q.max_x;
  c.max_y = q.max_y;
  c.have_left = hl;
  c.have_above = ha;
  c.bd = q.bd;
  const int va = lane < w ? c.above(lane) : 0, vl = lane < h ? c.left(lane) : 0;
  above[lane] = va;
  left[lane] = vl;
  wsync();
  int dc = 1 << (q.bd - 1);
  if (mode == 0 && (ha || hl)) {
    const int sum = wave_total((ha ? va : 0) + (hl ? vl : 0));
    dc = ha && hl ? (sum + ((w + h) >> 1)) / (w + h) : hl ? (sum + (h >> 1)) >> ilog2(h) : (sum + (w >> 1)) >> lw;
  }
  const int* sw = SPEC(AV1T_OFF_SM_WEIGHTS);
  for (int s = lane; s < w * h; s += 64) {
    const int x = s & (w - 1), y = s >> lw;
    int v = dc;
    if (mode == 1) {
      v = above[x];
    } else if (mode == 2) {
      v = left[y];
    } else if (mode == 3) {
      const int wy = sw[h - 4 + y], wx = sw[w - 4 + x];
      v = rnd2(wy * above[x] + (256 - wy) * left[h - 1] + wx * left[y] + (256 - wx) * above[w - 1], 9);
    }
    const int m = mask[s];
    pred[s] = (uint16_t)((m * v + (64 - m) * (int)pred[s] + 32) >> 6);
  }
  wsync();
}

__device__ void reconstruct_queued(RArgs a, BlkRef b, const QBlk& q, int* work, uint16_t* pred, const EarlyRes& er,
                                   const int* tab, uint32_t* error) {
  bool fused = false;
  if (q.kind == kIntra) {
    fused = predict_intra(a, b, q, work, pred, tab, er, error);
  } else if (q.flags & kInterDone) {
    ii_blend(b, q, work, pred);
  } else {
    /* inter/intra or intra block copy: reads the frame being decoded */
    const int lw = ilog2(b.w);
    for (int s = threadIdx.x; s < b.w * b.h; s += 64)
      pred[s] = (uint16_t)(q.flags & kIntraBC ? queue_inter<true>(&a, &b, s & (b.w - 1), s >> lw)
                                              : queue_inter<false>(&a, &b, s & (b.w - 1), s >> lw));
    wsync();
  }
  const int p = q.plane, stride = q.stride;
  if (er.on) {
    if (fused) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int s = threadIdx.x + 64 * k;
      if (s < q.w * q.h) pred[s] = (uint16_t)clampi((int)pred[s] + er.v[k], 0, q.maxv);
    }
    wsync();
    return;
  }
  for (int t = 0; t < b.tx_count; ++t) {
    const AV1H_CMEM DevTx& tx = cmem(a.plan.tx)[b.tx_first + t];
    const int ox = tx.x - b.x, oy = tx.y - b.y, ltw = ilog2(tx.w), n = tx.w * tx.h;
    const int16_t* r = a.res + a.lay.plane_off[p] + (int64_t)tx.y * stride + tx.x;
    /* eight residual loads in flight per lane before the first add */
    for (int s0 = threadIdx.x; s0 < n; s0 += 64 * 8) {
      int rv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int s = s0 + 64 * u;
        rv[u] = s < n ? r[(int64_t)(s >> ltw) * stride + (s & (tx.w - 1))] : 0;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int s = s0 + 64 * u;
        if (s < n) {
          uint16_t* q = pred + (oy + (s >> ltw)) * b.w + ox + (s & (tx.w - 1));
          *q = (uint16_t)clampi((int)*q + rv[u], 0, a.maxv);
        }
      }
    }
  }
  wsync();
}

/* Motion compensation, one 256 thread workgroup per task (at most 512
 * samples of consecutive items in coding order, an item being a block or a
 * row strip of a large one):
 *   A  a thread per item and one per item's reference turn the host's
 *      descriptors into what the passes read per lane (addresses, positions,
 *      places in LDS), with the item of every 16 samples and the reference of
 *      every 64 intermediates;
 *   B  the horizontal 8 tap pass over every reference row the item's
 *      vertical taps need, four columns per lane, the taps read from the
 *      reference and clamped to its visible area the way each tap is
 *      (av1gpu_kernels.h:1704-1711), rounded by InterRound0, into an LDS
 *      intermediate (16 bit: at most 200 * 4095 >> 5);
 *   C  per four output samples of a row: the vertical pass, InterRound1, the
 *      compound blend (av1gpu_kernels.h:2207-2293), one 8 byte store.
 * Bound by instructions and their latency, not bytes (a 1080p frame's 15 MB
 * of references and 7 MB of prediction are 5 us at the copy rate), so a lane
 * takes four neighbouring samples: their item is looked up once, an unscaled
 * row's eleven samples come in two loads and a scaled sample's eight in one,
 * and taps are multiplied two at a time (v_dot2_i32_i16: samples and taps are
 * 16 bit, sums below 2^31); 64 registers keep 8 workgroups on a compute unit.
 * A launch against one thread per sample: 720p frame 22.5 -> 12 us, 1080p
 * (scaled, compound) 45 -> 32, 2160p 169 -> 106, eight streams 122 -> 56. */
constexpr int kMcPairs = 2 * kMcItems;
constexpr int kMcChunkS = 16, kMcChunkM = 64; /* lookup: samples, intermediates */

/* one reference of an item, for the horizontal pass: its plane, the column
 * position of the first sample (stx 0: unscaled, in samples, else in 1/1024
 * with the step stx), its window's first row, its visible size, its filter row
 * (unscaled: with the phase) */
struct __align__(16) McPair {
  const AV1H_GLOBAL uint16_t* base;
  int stride, mid, lw, x0, stx, y0, rw, rh, taps, pad;
};
/* an item, for the vertical pass; of each reference, its intermediates and the
 * row position of its first row in them (1/1024) with the step */
struct __align__(16) McItem {
  AV1H_GLOBAL uint16_t* out;
  int stride, px0, lw, compound, w0, w1, taps, plane, ax, ay;
  struct {
    int mid, pos, step, pad;
  } r[2];
};
struct McLds {
  __align__(16) int16_t mid[kMcMid];
  McPair pair[kMcPairs];
  McItem item[kMcItems];
  int moff[kMcPairs + 1];
  uint8_t item_of[kMcSamples / kMcChunkS], pair_of[kMcMid / kMcChunkM];
};

__device__ void mc_body(RArgs a, int tn, const int16_t* s_filt, McLds& L_) {
  const int tid = threadIdx.x;
  const AV1H_CMEM McTaskDev& task = cmem(a.plan.mc_task)[tn];
  const int nit = task.count, npairs = 2 * nit, mtotal = task.mtotal, samples = task.samples;
  const PlaneVals<int> strides = plane_vals(a.lay.stride);
  const PlaneVals<int64_t> poffs = plane_vals(a.lay.plane_off);
  if (tid < npairs) {
    const McItemDev& it = a.plan.mc_items[task.first + (tid >> 1)];
    const McRefDev& q = it.r[tid & 1];
    McPair m;
    m.base = (const AV1H_GLOBAL uint16_t*)a.pool + (size_t)q.slot * a.slot_size + poffs[it.plane];
    m.stride = strides[it.plane];
    m.mid = q.mid_off;
    m.lw = ilog2(it.w);
    m.x0 = q.scaled ? q.sx0 : it.x + q.ix;
    m.stx = q.scaled ? q.stx : 0;
    m.y0 = q.wy0;
    m.rw = it.ref_w;
    m.rh = it.ref_h;
    m.taps = it.hk + (q.scaled ? 0 : q.fx * 8);
    m.pad = 0;
    L_.pair[tid] = m;
    L_.moff[tid] = m.mid;
    const int end = (tid & 1) < it.nref ? m.mid + q.wh * it.w : m.mid;
    for (int c = (m.mid + kMcChunkM - 1) / kMcChunkM; c * kMcChunkM < end; ++c) L_.pair_of[c] = (uint8_t)tid;
  } else if (tid >= 128 && tid < 128 + nit) {
    const int i = tid - 128;
    const McItemDev& it = a.plan.mc_items[task.first + i];
    McItem m;
    m.plane = it.plane;
    m.stride = strides[it.plane];
    m.ax = it.x;
    m.ay = it.y + it.y0;
    m.out = (AV1H_GLOBAL uint16_t*)a.frame + poffs[it.plane] + (int64_t)m.ay * m.stride + m.ax;
    m.px0 = it.px0;
    m.lw = ilog2(it.w);
    m.compound = it.compound;
    m.w0 = it.w0;
    m.w1 = it.w1;
    m.taps = it.vk;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const McRefDev& q = it.r[r];
      m.r[r].mid = q.mid_off;
      m.r[r].pos = q.scaled ? q.sy0 + q.sty * it.y0 - ((q.wy0 + 3) << 10) : q.fy << 6;
      m.r[r].step = q.scaled ? q.sty : 1024;
      m.r[r].pad = 0;
    }
    L_.item[i] = m;
    /* blocks hold multiples of 16 samples: a chunk lies in one item */
    for (int c = m.px0 / kMcChunkS; c * kMcChunkS < m.px0 + (it.rows << m.lw); ++c) L_.item_of[c] = (uint8_t)i;
  }
  if (tid == 0) L_.moff[npairs] = mtotal;
  __syncthreads();
  const int bd = a.lay.bit_depth;
  const int round0 = bd >= 12 ? 5 : 3;
  const int add0 = 1 << (round0 - 1);
  /* horizontal pass over every reference row an item needs, taps read from
   * the reference (clamped to it); block widths are multiples of 4, so the
   * four intermediates lie in one row */
  for (int e = tid * 4; e < mtotal; e += 1024) {
    int k = L_.pair_of[e / kMcChunkM];
    while (L_.moff[k + 1] <= e) ++k;
    const McPair q = L_.pair[k];
    const int o = e - q.mid, rr = o >> q.lw, x = o & ((1 << q.lw) - 1);
    const int y = clampi(q.y0 + rr, 0, q.rh - 1);
    const AV1H_GLOBAL uint16_t* row = q.base + (int64_t)y * q.stride;
    int v[4];
    if (!q.stx) {
      const int cx = q.x0 + x;
      const int4 f = *reinterpret_cast<const int4*>(s_filt + q.taps);
      uint32_t s[6];
      if (cx >= 3 && cx + 7 < q.rw) {
        /* cx - 3 .. cx + 7 (and one of the row's padding at its end) */
        load_words<4>(row + cx - 3, s);
        load_words<2>(row + cx + 5, s + 4);
      } else {
#pragma unroll
        for (int t = 0; t < 6; ++t)
          s[t] = pack2(row[clampi(cx - 3 + 2 * t, 0, q.rw - 1)], row[clampi(cx - 2 + 2 * t, 0, q.rw - 1)]);
      }
      uint32_t m[5]; /* the pairs in between */
#pragma unroll
      for (int t = 0; t < 5; ++t) m[t] = __builtin_amdgcn_alignbit(s[t + 1], s[t], 16);
      v[0] = dot8(s[0], s[1], s[2], s[3], f, add0);
      v[1] = dot8(m[0], m[1], m[2], m[3], f, add0);
      v[2] = dot8(s[1], s[2], s[3], s[4], f, add0);
      v[3] = dot8(m[1], m[2], m[3], m[4], f, add0);
    } else {
      uint32_t s[4][4];
      const int pos = q.x0 + q.stx * x;
      if ((pos >> 10) >= 3 && ((pos + 3 * q.stx) >> 10) + 4 < q.rw) {
#pragma unroll
        for (int i = 0; i < 4; ++i) load_words<4>(row + ((pos + i * q.stx) >> 10) - 3, s[i]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int cx = (pos + i * q.stx) >> 10;
#pragma unroll
          for (int t = 0; t < 4; ++t)
            s[i][t] = pack2(row[clampi(cx - 3 + 2 * t, 0, q.rw - 1)], row[clampi(cx - 2 + 2 * t, 0, q.rw - 1)]);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ph = ((pos + i * q.stx) & 1023) >> 6;
        v[i] = dot8(s[i][0], s[i][1], s[i][2], s[i][3], *reinterpret_cast<const int4*>(s_filt + q.taps + ph * 8), add0);
      }
    }
    uint2 out;
    out.x = pack2(v[0] >> round0, v[1] >> round0);
    out.y = pack2(v[2] >> round0, v[3] >> round0);
    *reinterpret_cast<uint2*>(L_.mid + e) = out;
  }
  __syncthreads();
  /* vertical pass and blend, four output samples of a row per lane */
  for (int si = tid * 4; si < samples; si += 1024) {
    const McItem& it = L_.item[L_.item_of[si / kMcChunkS]];
    const int s = si - it.px0, lw = it.lw, w = 1 << lw;
    const int x = s & (w - 1), ry = s >> lw;
    const int compound = it.compound;
    int round1 = compound ? 7 : 11;
    if (bd >= 12 && !compound) round1 -= 2;
    int v[2][4] = {};
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      if (r == 1 && !compound) break;
      const int pos = it.r[r].pos + it.r[r].step * ry;
      const int16_t* m = L_.mid + it.r[r].mid + ((pos >> 10) << lw) + x;
      const int4 f = *reinterpret_cast<const int4*>(s_filt + it.taps + ((pos & 1023) >> 6) * 8);
      const int ft[4] = {f.x, f.y, f.z, f.w};
      int acc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = 1 << (round1 - 1);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        /* two rows' columns side by side: low halves, high halves */
        const uint2 u = *reinterpret_cast<const uint2*>(m + ((2 * t) << lw));
        const uint2 d = *reinterpret_cast<const uint2*>(m + ((2 * t + 1) << lw));
        acc[0] = dot2(__builtin_amdgcn_perm(d.x, u.x, 0x05040100u), ft[t], acc[0]);
        acc[1] = dot2(__builtin_amdgcn_perm(d.x, u.x, 0x07060302u), ft[t], acc[1]);
        acc[2] = dot2(__builtin_amdgcn_perm(d.y, u.y, 0x05040100u), ft[t], acc[2]);
        acc[3] = dot2(__builtin_amdgcn_perm(d.y, u.y, 0x07060302u), ft[t], acc[3]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) v[r][i] = acc[i] >> round1;
    }
    const int post = 2 * 7 - (round0 + 7), w0 = it.w0, w1 = it.w1;
    int out[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int o = v[0][i];
      if (compound) {
        if (compound == AV1H_COMPOUND_AVERAGE)
          o = (v[0][i] + v[1][i] + (1 << post)) >> (1 + post);
        else
          o = (w0 * v[0][i] + w1 * v[1][i] + (1 << (3 + post))) >> (4 + post);
      }
      out[i] = clampi(o, 0, a.maxv);
    }
    *(AV1H_GLOBAL uint64_t*)(it.out + (int64_t)ry * it.stride + x) =
        (uint64_t)pack2(out[2], out[3]) << 32 | pack2(out[0], out[1]);
    /* the block's dependency cells (2 or 4 samples a side; blocks lie on
     * multiples of 4): final once the inter transforms after this launch have
     * run, which the queue launch follows */
    const int p = it.plane, sh = plane_vals(a.lay.cell_shift)[p], ax = it.ax + x, ay = it.ay + ry;
    if (a.plan.cell_waits && (ay & ((1 << sh) - 1)) == 0) {
      const int cw = plane_vals(a.lay.cells_w)[p], cy = ay >> sh;
      uint32_t* cells = a.cells + plane_vals(a.lay.cell_off)[p] + (int64_t)cy * cw;
      for (int cx = ax >> sh; cx << sh < ax + 4; ++cx)
        if (cx < cw && cy < plane_vals(a.lay.cells_h)[p]) cells[cx] = a.epoch;
    }
  }
}

__global__ __launch_bounds__(256, 8) void k_mc(BatchDev B) {
  __shared__ __align__(16) int16_t s_filt[768];
  __shared__ McLds s_lds;
  for (int i = threadIdx.x; i < 768; i += 256) s_filt[i] = (int16_t)av1t_spec_table[AV1T_OFF_SUBPEL + i];
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKMc);
  const int total = pre[B.njobs];
  for (int base = 0; base < total; base += gridDim.x) {
    const int v = xcd_group(base, total);
    if (v < 0) continue;
    const int j = find_job(pre, B.njobs, v);
    mc_body(recon_args(B, j), v - pre[j], s_filt, s_lds);
    __syncthreads();
  }
}

/* Inter blocks with warp, masks or OBMC, and the inter half of inter/intra
 * blocks (all read only references): the direct per sample computation, a
 * sample's eight rows loaded together. kSpecialStrips waves share a block: with
 * one, the launch is as long as the largest block; with 16, most of them find
 * no sample. 853x479 frame of these tools: 249 us with one load after another
 * and one wave a block, 117 with 16 waves, 63 with four. */
__global__ __launch_bounds__(64) void k_inter_special(BatchDev B) {
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKSpecial);
  const int total = pre[B.njobs];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int j = find_job(pre, B.njobs, v);
    RArgs a = recon_args(B, j);
    const int strip = (v - pre[j]) % kSpecialStrips;
    const int bi = cmem(a.plan.special_list)[(v - pre[j]) / kSpecialStrips];
    BlkRef b = cmem(a.plan.blocks)[bi];
    const int p = b.plane, stride = a.lay.stride[p], lw = ilog2(b.w);
    uint16_t* dst = a.frame + a.lay.plane_off[p] + (size_t)b.y * stride + b.x;
    for (int s = strip * 64 + threadIdx.x; s < b.w * b.h; s += 64 * kSpecialStrips)
      dst[(size_t)(s >> lw) * stride + (s & (b.w - 1))] = (uint16_t)inter_sample<false>(a, b, s & (b.w - 1), s >> lw);
    if (strip == 0 && a.plan.cell_waits && !(b.flags & kInterIntra)) mark_cells(a, b, false);
  }
}

/* Every block the two paths above do not take (CFL, palette, filter intra,
 * several transforms, inter/intra, intra block copy, edges that need the cell
 * wait), from its wait to its stores; returns when it was ready. A call of its
 * own: inlined, its registers (above 256) halved the kernel's waves and its
 * spills lay in the way of every block (queue of a 1080p key frame 762 -> 992
 * us). */
__device__ __noinline__ uint64_t queue_general(const AV1H_CMEM ReconArgs* args, const AV1H_CMEM DevBlock* block,
                                               AV1H_LDS int* lds_work, AV1H_LDS uint16_t* lds_pred,
                                               AV1H_LDS const int* lds_tab, uint32_t* error, bool trace) {
  /* arguments come in vector registers: these are the same in every lane */
  RArgs a = *(const AV1H_CMEM ReconArgs*)sreg((int64_t)args);
  BlkRef b = *(const AV1H_CMEM DevBlock*)sreg((int64_t)block);
  int* work = (int*)lds_work;
  uint16_t* pred = (uint16_t*)lds_pred;
  const int* tab = (const int*)lds_tab;
  const EarlyRes er = early_residual(a, b, one_transform(a, b));
  const QBlk q = queued_block(a, b);
  if (q.flags & kInterDone) ii_ahead(a, b, q, work, pred);
  if (b.flags & kPackedEdges)
    gather_edges(a, b, work, error);
  else
    wait_cells(a, b, error);
  const uint64_t ready = trace ? (uint64_t)wall_clock64() : 0;
  reconstruct_queued(a, b, q, work, pred, er, tab, error);
  /* the packed edges first: the blocks waiting on this one read only them */
  if (q.flags & (kEdgeRow | kEdgeCol)) write_edges(q, pred);
  store_block(q, pred);
  return ready;
}

__global__ __launch_bounds__(64) void k_queue(BatchDev B) {
  __shared__ int s_work[kWork];
  __shared__ uint16_t s_pred[64 * 64];
  __shared__ int s_tab[kTabHi - kTabLo];
  const int nqueue = kernel_prefix(B, kKernels)[0];
  /* more workgroups than entries: the rest leave without the device-scope
   * atomic each would make on the one counter (with the small blocks' path,
   * a 160x96 inter frame's queue of 27 blocks 28.8 -> 8.9 us) */
  const int takers = min((int)gridDim.x, nqueue);
  if ((int)blockIdx.x >= takers) return;
  for (int i = threadIdx.x; i < kTabHi - kTabLo; i += 64) s_tab[i] = av1t_spec_table[kTabLo + i];
  __syncthreads();
  /* Tickets: atomics on one address are served one after another (11.4 ns
   * each: 17 us for the first tickets of 1536 waves, with their descriptor
   * loads stuck behind them), so a large queue is dealt to kTickets counters,
   * entry idx to counter idx % kTickets. Every entry still gets a wave: an
   * XCD's workgroups start in order of their number, the first kTickets of
   * them on any XCD cover every counter, and a counter's waves take its
   * entries in order, so the smallest unfinished entry is held by a wave or
   * next on a counter with a wave that holds none. That takes kTickets resident
   * workgroups on one XCD (with one counter, one in all): a compute unit holds
   * eight of this kernel (227 registers, 28 bytes of scratch a lane: two waves a
   * SIMD; 18 KB of LDS), an XCD 256, so of up to 32 such launches at a time (a
   * process has four hardware queues) one has them even where waiting waves
   * fill the card, and when it ends its places go to the next. Queue of a 1080p inter
   * frame (2518 entries) 67 -> 42 us, of a batch of eight (12,400) 169 -> 61. */
  const int deal = takers >= 16 * kTickets ? kTickets : 1;
  const int own = ((int)blockIdx.x >> 3) & (deal - 1);
  const int own_n = (nqueue - own + deal - 1) / deal; /* entries and takers of this counter */
  const int own_takers = deal == 1 ? takers : takers / (8 * deal) * 8 + clampi(takers % (8 * deal) - 8 * own, 0, 8);
  uint32_t* counter = B.queue_counter + own * kTicketStep;
  for (;;) {
    int ticket = 0;
    if (threadIdx.x == 0) ticket = (int)atomicAdd(counter, 1u);
    ticket = __builtin_amdgcn_readfirstlane(ticket);
    if (ticket >= own_n) {
      /* every taking workgroup takes exactly one ticket past the end; the last of
       * those is the counter's last use in this launch, so it resets the
       * counter for the next one */
      if (threadIdx.x == 0 && ticket == own_n + own_takers - 1)
        __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    const int idx = ticket * deal + own;
    const uint64_t t0 = B.trace ? (uint64_t)wall_clock64() : 0;
    int job = 0, blk;
    if (B.queue) {
      const uint32_t e = cmem(B.queue)[idx];
      job = (int)(e >> kQueueJobShift);
      blk = (int)(e & ((1u << kQueueJobShift) - 1));
    } else {
      blk = cmem(recon_args(B, 0).plan.queue_list)[idx];
    }
    RArgs a = recon_args(B, __builtin_amdgcn_readfirstlane(job));
    BlkRef b = cmem(a.plan.blocks)[__builtin_amdgcn_readfirstlane(blk)];
    const bool one = one_transform(a, b);
    const QBlk q = queued_block(a, b);
    uint64_t t1 = 0;
    if (small_block(q, b, one)) {
      queue_small(a, b, q, one, s_tab, B.error, &t1, B.trace != nullptr);
    } else if (big_block(q, b, one)) {
      queue_big(a, b, q, one, s_work, s_tab, B.error, &t1, B.trace != nullptr);
    } else {
      t1 = queue_general(&a, &b, (AV1H_LDS int*)s_work, (AV1H_LDS uint16_t*)s_pred, (AV1H_LDS const int*)s_tab, B.error,
                         B.trace != nullptr);
    }
    if (!(q.flags & kSkipMark)) {
      /* every sample store of the block has completed before its cells flip */
      __builtin_amdgcn_s_waitcnt(0);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      mark_cells(a, b, true);
    }
    wsync();
    if (B.trace && threadIdx.x == 0) {
      /* diagnostics: when the block was taken, found ready, published */
      uint64_t* t = B.trace + 4 * (size_t)idx;
      t[0] = t0;
      t[1] = t1;
      t[2] = (uint64_t)wall_clock64();
      t[3] = (uint64_t)blockIdx.x;
    }
  }
}


}  // namespace

int itx_groups(const FramePlanDev& p, int set, int c0, int c1) {
  int g = 0;
  for (int c = c0; c < c1; ++c) {
    const int n = p.itx_off[set][c + 1] - p.itx_off[set][c], per = 16 >> c;
    g += (n + per - 1) / per;
  }
  return g;
}

hipError_t launch_recon_kernel(const BatchDev& b, int k, int total, int cap, hipStream_t s) {
  const dim3 grid(min(total, cap));
  switch (k) {
    case kKMc: hipLaunchKernelGGL(k_mc, grid, dim3(256), 0, s, b); break;
    case kKSpecial: hipLaunchKernelGGL(k_inter_special, grid, dim3(64), 0, s, b); break;
    /* both sets of transforms in one launch: `total` counts both */
    case kKItxInter: hipLaunchKernelGGL((k_itx<0, 3>), grid, dim3(64), 0, s, b); break;
    case kKItxInterL: hipLaunchKernelGGL((k_itx<3, 5>), grid, dim3(64), 0, s, b); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_queue(const BatchDev& b, int total, int cap, hipStream_t s, int* launches) {
  if (total == 0) return hipSuccess;
  const int grid = total < 0 ? cap : min(total, cap);
  hipLaunchKernelGGL(k_queue, dim3(grid), dim3(64), 0, s, b);
  *launches += 1;
  return hipGetLastError();
}

}  // namespace av1hip
