/*
 * Post-reconstruction passes for gfx950: deblocking (two ordered passes),
 * CDEF, superres upscaling, loop restoration, and the NV12 / RGB packs. The
 * arithmetic is the reference's (kernels/av1gpu_kernels.h), cited per function.
 */
#define AV1T_TABLE_QUAL static __constant__ const
#include "av1hip_internal.hpp"
#include "spec_tables.h"

#include <climits>

namespace av1hip {
namespace {

#define SPEC(off) (av1t_spec_table + (off))

/* global (not generic) pointers: their accesses need no wait for LDS */
#define AV1H_GLOBAL __attribute__((address_space(1)))

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }
__device__ __forceinline__ int rnd2(int v, int n) { return n <= 0 ? v : (v + (1 << (n - 1))) >> n; }
__device__ __forceinline__ int rsr64(int64_t v, int n) { return (int)((v + ((int64_t)1 << (n - 1))) >> n); }

/* ---- deblocking (av1gpu_kernels.h:2422-2572) --------------------------- */

__device__ __forceinline__ int f4c(int v, int bd) { return clampi(v, -(1 << (bd - 1)), (1 << (bd - 1)) - 1); }

/* The flat filters: outputs p(N-1)..q(N-1) from taps p(N)..q(N), the centre
 * N2 taps weighted twice, all indices fixed at compile time
 * (av1gpu_kernels.h:2540-2568). v[j] holds the sample at b[(j - 5) s]. */
template <int N, int N2, int LG>
__device__ __forceinline__ void wide_filter(const int* v, uint16_t* b, int s, int maxv) {
  int res[2 * N];
#pragma unroll
  for (int i = -N; i < N; ++i) {
    int t = 0;
#pragma unroll
    for (int k = -N; k <= N; ++k) {
      const int idx = i + k < -(N + 1) ? -(N + 1) : (i + k > N ? N : i + k);
      t += v[idx + 7] * ((k <= N2 && k >= -N2) ? 2 : 1);
    }
    res[i + N] = rnd2(t, LG);
  }
#pragma unroll
  for (int i = -N; i < N; ++i) b[(2 + i) * s] = (uint16_t)clampi(res[i + N], 0, maxv);
}

/* one line across one edge: b points at p1, s is the step across the edge.
 * Every sample the line's filter size can use is loaded first, together, so
 * the decisions do not wait on one load after another. */
__device__ void deblock_line(uint16_t* b, int s, int level, int sharp, int fs, int chroma, int bd,
                             int maxv) {
  const int sh = bd - 8, mid = 0x80 << sh;
  const int flen = fs == 4 ? 4 : (chroma ? 6 : (fs == 8 ? 8 : 16));
  /* v[j] = b[(j - 5) s]: p6 .. p1 at 0 .. 5, p0 6, q0 7, q1 .. q6 at 8 .. 13 */
  const int jlo = fs >= 16 ? 0 : (flen >= 8 ? 3 : (flen >= 6 ? 4 : 5));
  const int jhi = fs >= 16 ? 13 : (flen >= 8 ? 10 : (flen >= 6 ? 9 : 8));
  int v[14];
#pragma unroll
  for (int j = 0; j < 14; ++j) v[j] = (j >= jlo && j <= jhi) ? (int)b[(j - 5) * s] : 0;
  const int p1 = v[5], p0 = v[6], q0 = v[7], q1 = v[8];
  const int lsh = sharp > 4 ? 2 : (sharp > 0 ? 1 : 0);
  int limit = level >> lsh;
  if (limit < 1) limit = 1;
  if (sharp > 0 && limit > 9 - sharp) limit = 9 - sharp;
  const int blim = (2 * (level + 2) + limit) << sh, lim = limit << sh, thr = (level >> 4) << sh;
  const int one = 1 << sh;
  const int hev = abs(p1 - p0) > thr || abs(q1 - q0) > thr;
  int bad = abs(p1 - p0) > lim || abs(q1 - q0) > lim || abs(p0 - q0) * 2 + abs(p1 - q1) / 2 > blim;
  const int p2 = v[4], q2 = v[9], p3 = v[3], q3 = v[10];
  if (flen >= 6) bad = bad || abs(p2 - p1) > lim || abs(q2 - q1) > lim;
  if (flen >= 8) bad = bad || abs(p3 - p2) > lim || abs(q3 - q2) > lim;
  if (bad) return;
  int flat = 1, flat2 = 1;
  if (fs >= 8) {
    int f = abs(p1 - p0) > one || abs(q1 - q0) > one || abs(p2 - p0) > one || abs(q2 - q0) > one;
    if (flen >= 8) f = f || abs(p3 - p0) > one || abs(q3 - q0) > one;
    flat = !f;
  }
  if (fs >= 16) {
    flat2 = !(abs(v[0] - p0) > one || abs(v[13] - q0) > one || abs(v[1] - p0) > one || abs(v[12] - q0) > one ||
              abs(v[2] - p0) > one || abs(v[11] - q0) > one);
  }
  if (fs == 4 || !flat) {
    const int ps1 = p1 - mid, ps0 = p0 - mid, qs0 = q0 - mid, qs1 = q1 - mid;
    int f = hev ? f4c(ps1 - qs1, bd) : 0;
    f = f4c(f + 3 * (qs0 - ps0), bd);
    const int f1 = f4c(f + 4, bd) >> 3, f2 = f4c(f + 3, bd) >> 3;
    b[2 * s] = (uint16_t)clampi(f4c(qs0 - f1, bd) + mid, 0, maxv);
    b[s] = (uint16_t)clampi(f4c(ps0 + f2, bd) + mid, 0, maxv);
    if (!hev) {
      const int f3 = rnd2(f1, 1);
      b[3 * s] = (uint16_t)clampi(f4c(qs1 - f3, bd) + mid, 0, maxv);
      b[0] = (uint16_t)clampi(f4c(ps1 + f3, bd) + mid, 0, maxv);
    }
    return;
  }
  if (fs >= 16 && flat2)
    wide_filter<6, 1, 4>(v, b, s, maxv);
  else if (chroma)
    wide_filter<2, 1, 3>(v, b, s, maxv);
  else
    wide_filter<3, 0, 3>(v, b, s, maxv);
}

/* One thread per line; edges of one direction never share samples. The edge
 * owning line g is found from the first edge of the thread's 256 line chunk
 * (a table the host builds) and a short forward scan. */
__device__ void deblock_chunk(FArgs a, int first, int count, int lines, const int32_t* chunk,
                              int ci, int* s_line0) {
  /* the chunk's lines lie in the 256 edges from its first one (an edge
   * covers at least one line): their first lines go to LDS, and every
   * thread finds its edge by binary search there */
  const DevDeblock* edges = a.plan.deblock + first;
  const int e0 = chunk[ci], ne = min(count - e0, 256);
  if ((int)threadIdx.x < ne) s_line0[threadIdx.x] = edges[e0 + threadIdx.x].line0;
  __syncthreads();
  const int g = ci * 256 + threadIdx.x;
  if (g >= lines) return;
  int lo = 0, hi = ne - 1;
  while (lo < hi) {
    const int m = (lo + hi + 1) >> 1;
    if (s_line0[m] <= g)
      lo = m;
    else
      hi = m - 1;
  }
  const DevDeblock& e = edges[e0 + lo];
  if (e.level == 0) return;
  const int k = g - e.line0;
  const int p = e.plane_vertical & 3, st = a.lay.stride[p];
  uint16_t* plane = a.frame + a.lay.plane_off[p];
  uint16_t* b;
  int s;
  if (e.plane_vertical & 4) {
    b = plane + (size_t)(e.y + k) * st + (e.x - 2);
    s = 1;
  } else {
    b = plane + (size_t)(e.y - 2) * st + (e.x + k);
    s = st;
  }
  deblock_line(b, s, e.level, a.sharpness, e.filter_size, p != 0, a.lay.bit_depth, a.maxv);
}

/* the vertical edges (pass 0) or the horizontal edges (pass 1) of every frame */
__global__ __launch_bounds__(256) void k_deblock(BatchDev B, int pass) {
  __shared__ int s_line0[256];
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, (pass ? kKDeblockH : kKDeblockV));
  const int total = pre[B.njobs];
  for (int base = 0; base < total; base += gridDim.x) {
    const int v = xcd_group(base, total);
    if (v < 0) continue;
    const int j = find_job(pre, B.njobs, v);
    FArgs a = filter_args(B, j);
    PlanRef P = a.plan;
    if (pass)
      deblock_chunk(a, P.n_deblock_v, P.n_deblock_h, P.lines_h, P.db_chunk + (P.lines_v + 255) / 256, v - pre[j],
                    s_line0);
    else
      deblock_chunk(a, 0, P.n_deblock_v, P.lines_v, P.db_chunk, v - pre[j], s_line0);
    __syncthreads();
  }
}

/* ---- CDEF (av1gpu_kernels.h:2601-2775) ---------------------------------- */

__device__ __forceinline__ int flog2(int v) { return 31 - __builtin_clz(v); }

/* Direction search of luma 8x8 blocks (av1gpu_kernels.h:2601-2660), one
 * block per lane: a lane reads its block's eight rows (one 16-byte load
 * each: rows start on 8-sample boundaries of 128-sample aligned strides),
 * keeps the eight directions' line sums in registers (every index a
 * compile-time constant), weighs them and picks the first direction of
 * largest cost. No LDS and no cross-lane traffic: consecutive lanes take
 * consecutive listed blocks, so a wave's row loads cover whole 128-byte
 * spans of a block row. Writes (direction, variance) for each block into
 * `dirmap`. */
__device__ __forceinline__ void cdef_dir_block(FArgs a, int bi) {
  const int pos = a.plan.cdef_dir_list[bi];
  const int bx = pos & 0xffff, by = pos >> 16;
  const int sh = a.lay.bit_depth - 8;
  const uint16_t* src = a.cdef_src + a.lay.plane_off[0] + (size_t)(by * 8) * a.lay.stride[0] + bx * 8;
  int p0[15] = {}, p1[11] = {}, p2[8] = {}, p3[11] = {}, p4[15] = {}, p5[11] = {}, p6[8] = {}, p7[11] = {};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint4 r = *reinterpret_cast<const uint4*>(src + (size_t)i * a.lay.stride[0]);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int x = (int)(((w[k >> 1] >> (16 * (k & 1))) & 0xffffu) >> sh) - 128;
      p0[i + k] += x;
      p1[i + k / 2] += x;
      p2[i] += x;
      p3[3 + i - k / 2] += x;
      p4[7 + i - k] += x;
      p5[3 - i / 2 + k] += x;
      p6[k] += x;
      p7[i / 2 + k] += x;
    }
  }
  /* 840 / n for a line of n samples */
  constexpr int div[9] = {0, 840, 420, 280, 210, 168, 140, 120, 105};
  auto full = [&](const int* q) {
    int c = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) c += q[t] * q[t];
    return c * div[8];
  };
  auto diag = [&](const int* q) {
    int c = 0;
#pragma unroll
    for (int t = 0; t < 7; ++t) c += (q[t] * q[t] + q[14 - t] * q[14 - t]) * div[t + 1];
    return c + q[7] * q[7] * div[8];
  };
  auto half = [&](const int* q) {
    int c = 0;
#pragma unroll
    for (int t = 0; t < 5; ++t) c += q[3 + t] * q[3 + t];
    c *= div[8];
#pragma unroll
    for (int t = 0; t < 3; ++t) c += (q[t] * q[t] + q[10 - t] * q[10 - t]) * div[2 * t + 2];
    return c;
  };
  const int cost[8] = {diag(p0), half(p1), full(p2), half(p3), diag(p4), half(p5), full(p6), half(p7)};
  /* the first direction with the largest cost (a strict > scan from 0); a
   * block whose costs are all zero keeps direction 0 */
  int best = 0, dd = 0;
#pragma unroll
  for (int d = 0; d < 8; ++d)
    if (cost[d] > best) {
      best = cost[d];
      dd = d;
    }
  int opp = cost[0];
#pragma unroll
  for (int d = 1; d < 8; ++d)
    if (d == ((dd + 4) & 7)) opp = cost[d];
  int* m = a.cdef_dir + 2 * (by * a.cdef_dir_w + bx);
  m[0] = dd;
  m[1] = (best - opp) >> 10;
}

__global__ __launch_bounds__(256) void k_cdef_dir(BatchDev B) {
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKCdefDir);
  const int total = pre[B.njobs];
  for (int base = 0; base < total; base += gridDim.x) {
    const int v = xcd_group(base, total);
    if (v < 0) continue;
    const int j = find_job(pre, B.njobs, v);
    FArgs a = filter_args(B, j);
    const int bi = (v - pre[j]) * kCdefDirPerGroup + (int)threadIdx.x;
    if (bi < a.plan.n_cdef_dir) cdef_dir_block(a, bi);
  }
}

/* CDEF of the listed blocks (av1gpu_kernels.h:2662-2775), four neighbouring
 * samples of a block row per lane: a wave holds four luma blocks, four to
 * sixteen chroma blocks by subsampling. A lane reads its samples and each of
 * its twelve taps straight from the deblocked snapshot, three whole words that
 * hold them (loads that start inside a word ran at a fraction of the rate: 57
 * us on a 2160p frame instead of 48), and filters two samples per instruction
 * in packed 16-bit words. A tap outside the plane reads as
 * kCdefOutside, which is no minimum without a sign, no maximum with one, and so
 * far from every sample that its constrained difference is 0. Samples of
 * unlisted blocks are already final in the frame.
 * One sample per lane from LDS tiles, bound by instructions, took 24.5 us on a
 * 1080p frame, 79 on a 2160p one, 92 on eight streams; now 21, 43 and 53,
 * bound by the cache lines the loads touch: eight samples per lane halved the
 * instructions per sample and took 23, 56 and 66. */
typedef short cdef_s2 __attribute__((ext_vector_type(2)));
typedef unsigned short cdef_u2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kCdefOutside = 0x80008000u;

/* (dy, dx) of direction d's near and far tap: signed nibble d */
constexpr uint32_t kCdefDy0 = 0x1111000fu, kCdefDx0 = 0x00011111u, kCdefDy1 = 0x222210feu, kCdefDx1 = 0xf0122222u;
__device__ __forceinline__ int cdef_nibble(uint32_t table, int d) { return __builtin_amdgcn_sbfe((int)table, 4 * d, 4); }

/* one chroma direction for a luma one where the axes are scaled apart */
__device__ __forceinline__ int cdef_uv_dir(int ss_x, int ss_y, int d) {
  if (ss_x == ss_y) return d;
  return (int)((ss_x ? 0x66654207u : 0x06432221u) >> (4 * d)) & 7;
}

struct CdefPlane {
  const AV1H_GLOBAL uint16_t* src; /* the plane in the snapshot */
  int stride, w, h;
};

/* four samples from (x, y) on; with kEdge they may lie outside the plane, at
 * most two samples away (w is at least 4, a lane's own samples are inside) */
template <bool kEdge>
__device__ __forceinline__ uint2 cdef_load(const CdefPlane& P, int x, int y) {
  const int xa = kEdge ? clampi(x, 0, P.w - 4) : x, ya = kEdge ? clampi(y, 0, P.h - 1) : y;
  const int at = ya * P.stride + xa;
  const AV1H_GLOBAL uint32_t* q = (const AV1H_GLOBAL uint32_t*)(P.src + (at & ~1));
  const uint32_t w0 = q[0], w1 = q[1], w2 = q[2];
  uint2 v = make_uint2(__builtin_amdgcn_alignbit(w1, w0, (at & 1) * 16), __builtin_amdgcn_alignbit(w2, w1, (at & 1) * 16));
  if (kEdge) {
    const int n = x - xa;
    if (n < 0) {
      v.y = n == -1 ? __builtin_amdgcn_alignbit(v.y, v.x, 16) : v.x;
      v.x = n == -1 ? __builtin_amdgcn_alignbit(v.x, kCdefOutside, 16) : kCdefOutside;
    } else if (n > 0) {
      v.x = n == 1 ? __builtin_amdgcn_alignbit(v.y, v.x, 16) : v.y;
      v.y = n == 1 ? __builtin_amdgcn_alignbit(kCdefOutside, v.y, 16) : kCdefOutside;
    }
    if (y != ya) v = make_uint2(kCdefOutside, kCdefOutside);
  }
  return v;
}

struct CdefSum {
  cdef_s2 x[2], sum[2], hi[2];
  cdef_u2 lo[2];
};

/* one tap of weight wt: constrain() of its difference is the difference
 * clamped to +-max(0, thr - (|difference| >> adj)) */
__device__ __forceinline__ void cdef_add(CdefSum& s, uint2 v, uint32_t thr, uint32_t adj, uint32_t wt) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t w = i ? v.y : v.x;
    const cdef_s2 d = __builtin_bit_cast(cdef_s2, w) - s.x[i];
    const cdef_u2 mag = __builtin_bit_cast(cdef_u2, __builtin_elementwise_max(d, -d));
    const cdef_s2 lim = __builtin_bit_cast(
        cdef_s2, __builtin_elementwise_sub_sat(__builtin_bit_cast(cdef_u2, thr), mag >> __builtin_bit_cast(cdef_u2, adj)));
    s.sum[i] += __builtin_bit_cast(cdef_s2, wt) * __builtin_elementwise_max(__builtin_elementwise_min(d, lim), -lim);
  }
}

__device__ __forceinline__ void cdef_range(CdefSum& s, uint2 v) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    s.lo[i] = __builtin_elementwise_min(s.lo[i], __builtin_bit_cast(cdef_u2, i ? v.y : v.x));
    s.hi[i] = __builtin_elementwise_max(s.hi[i], __builtin_bit_cast(cdef_s2, i ? v.y : v.x));
  }
}

struct CdefTaps {
  int dir, pri, sec, adjp, adjs, pt0, pt1;
};

/* The result of one strength alone lies between the samples it weighs (12
 * sixteenths of their differences), so the other's taps, which only the range
 * needs, are left out then. */
template <bool kEdge>
__device__ __forceinline__ uint2 cdef_quad(const CdefPlane& P, int x, int y, const CdefTaps& c, int maxv) {
  const uint2 own = cdef_load<false>(P, x, y);
  CdefSum s;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    s.x[i] = s.hi[i] = __builtin_bit_cast(cdef_s2, i ? own.y : own.x);
    s.lo[i] = __builtin_bit_cast(cdef_u2, i ? own.y : own.x);
    s.sum[i] = cdef_s2{0, 0};
  }
  const bool both = c.pri != 0 && c.sec != 0;
  /* the primary direction and the two secondary ones; one copy of the code */
#pragma unroll 1
  for (int k = 0; k < 3; ++k) {
    if ((k ? c.sec : c.pri) == 0) continue;
    const int d = (c.dir + 2 * k + (k == 2 ? 2 : 0)) & 7;
    const int dx0 = cdef_nibble(kCdefDx0, d), dy0 = cdef_nibble(kCdefDy0, d);
    const int dx1 = cdef_nibble(kCdefDx1, d), dy1 = cdef_nibble(kCdefDy1, d);
    const uint32_t thr = (k ? c.sec : c.pri) * 0x10001u, adj = (k ? c.adjs : c.adjp) * 0x10001u;
    const uint32_t w0 = (k ? 2 : c.pt0) * 0x10001u, w1 = (k ? 1 : c.pt1) * 0x10001u;
    const uint2 v[4] = {cdef_load<kEdge>(P, x - dx0, y - dy0), cdef_load<kEdge>(P, x + dx0, y + dy0),
                        cdef_load<kEdge>(P, x - dx1, y - dy1), cdef_load<kEdge>(P, x + dx1, y + dy1)};
#pragma unroll
    for (int t = 0; t < 4; ++t) cdef_add(s, v[t], thr, adj, t < 2 ? w0 : w1);
    if (both) {
#pragma unroll
      for (int t = 0; t < 4; ++t) cdef_range(s, v[t]);
    }
  }
  uint32_t out[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    cdef_s2 f = s.x[i] + ((s.sum[i] + (s.sum[i] >> 15) + (short)8) >> 4);
    if (both) f = __builtin_elementwise_min(__builtin_elementwise_max(f, __builtin_bit_cast(cdef_s2, s.lo[i])), s.hi[i]);
    out[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(f, cdef_s2{(short)maxv, (short)maxv}));
  }
  return make_uint2(out[0], out[1]);
}

/* the same for strengths and dampings whose sums or shifts leave 16 bits (no
 * stream codes them): one sample and one tap at a time */
__device__ __forceinline__ uint2 cdef_quad_wide(const CdefPlane& P, int x, int y, const CdefTaps& c, int maxv) {
  uint32_t out[4];
#pragma unroll 1
  for (int i = 0; i < 4; ++i) {
    const int own = P.src[y * P.stride + x + i];
    int sum = 0, lo = own, hi = own;
#pragma unroll 1
    for (int t = 0; t < 12; ++t) {
      const int kind = (t >> 1) % 3, far = t >= 6;
      const int d = (c.dir + (kind == 0 ? 0 : kind == 1 ? 2 : 6)) & 7;
      int dy = cdef_nibble(far ? kCdefDy1 : kCdefDy0, d), dx = cdef_nibble(far ? kCdefDx1 : kCdefDx0, d);
      if (t & 1) dy = -dy, dx = -dx;
      const int tx = x + i + dx, ty = y + dy;
      if (tx < 0 || ty < 0 || tx >= P.w || ty >= P.h) continue;
      const int v = P.src[ty * P.stride + tx], mag = abs(v - own);
      const int con = max(0, min((kind ? c.sec : c.pri) - (mag >> (kind ? c.adjs : c.adjp)), mag));
      sum += (kind ? 2 - far : far ? c.pt1 : c.pt0) * (v < own ? -con : con);
      lo = min(lo, v);
      hi = max(hi, v);
    }
    const uint32_t r = clampi(clampi(own + ((8 + sum - (sum < 0)) >> 4), lo, hi), 0, maxv);
    out[0] = i == 0 ? r : out[0], out[1] = i == 1 ? r : out[1], out[2] = i == 2 ? r : out[2], out[3] = r;
  }
  return make_uint2(out[0] | out[1] << 16, out[2] | out[3] << 16);
}

/* the lane's four samples of set `grp` of blocks first .. first + count - 1 */
__device__ __forceinline__ void cdef_lane(FArgs a, int first, int count, int grp, bool luma) {
  LayRef L = a.lay;
  const int ss_x = luma ? 0 : L.ss_x, ss_y = luma ? 0 : L.ss_y;
  const int lanes = 4 - ss_x - ss_y; /* log2 of a block's lanes */
  const int bi = (grp << (8 - lanes)) + ((int)threadIdx.x >> lanes);
  if (bi >= count) return;
  const uint2 rec = *reinterpret_cast<const uint2*>(a.plan.cdef + first + bi);
  const int bx = (int)(rec.x & 0xffffu), by = (int)(rec.x >> 16);
  const int p = luma ? 0 : (int)(rec.y >> 16) & 3, cs = L.bit_depth - 8;
  CdefTaps c;
  c.pri = (int)(rec.y & 0xffu) << cs;
  c.sec = (int)((rec.y >> 8) & 0xffu) << cs;
  const int damping = (int)((rec.y >> 18) & 0x3fu) + cs - (luma ? 0 : 1);
  c.dir = (int)rec.y >> 24;
  if (c.dir < 0) {
    const int2 m = *reinterpret_cast<const int2*>(
        a.cdef_dir + 2 * (((by << ss_y) >> 3) * a.cdef_dir_w + ((bx << ss_x) >> 3)));
    c.dir = c.pri == 0 ? 0 : cdef_uv_dir(ss_x, ss_y, m.x);
    if (luma) {
      const int vs = (m.y >> 6) ? min(flog2(m.y >> 6), 12) : 0;
      c.pri = m.y ? ((c.pri * (4 + vs) + 8) >> 4) : 0;
    }
  }
  if (c.pri == 0 && c.sec == 0) return; /* the destination already holds the snapshot's values */
  c.adjp = c.pri ? max(0, damping - flog2(c.pri)) : 0;
  c.adjs = c.sec ? max(0, damping - flog2(c.sec)) : 0;
  const int ts = (c.pri >> cs) & 1;
  c.pt0 = ts ? 3 : 4;
  c.pt1 = ts ? 3 : 2;
  CdefPlane P;
  P.src = (const AV1H_GLOBAL uint16_t*)(a.cdef_src + L.plane_off[p]);
  P.stride = L.stride[p];
  P.w = L.grid_w[p];
  P.h = L.grid_h[p];
  const int l = (int)threadIdx.x & ((1 << lanes) - 1);
  const int x = bx + 4 * (l & (1 - ss_x)), y = by + (l >> (1 - ss_x));
  uint2 v;
  /* the weighted sum stays below 12 (pri + sec), a threshold shifted up by
   * its adjustment below 1 << (damping + 1): 2^15 and 28672 (the distance of
   * kCdefOutside from a sample) are out of reach */
  if (12 * (c.pri + c.sec) >= 32752 || damping > 13)
    v = cdef_quad_wide(P, x, y, c, a.maxv);
  else if (x < 2 || y < 2 || x + 6 > P.w || y + 3 > P.h)
    v = cdef_quad<true>(P, x, y, c, a.maxv);
  else
    v = cdef_quad<false>(P, x, y, c, a.maxv);
  const int64_t at = L.plane_off[p] + y * P.stride + x;
  *reinterpret_cast<uint2*>(a.cdef_dst + at) = v;
  if (a.cdef_dst2) *reinterpret_cast<uint2*>(a.cdef_dst2 + at) = v;
}

/* The luma blocks (plane 0) and then the chroma blocks (planes 1 and 2) of
 * every frame in one launch: the luma groups of every frame come first, then
 * the chroma groups (both read the deblocked snapshot and the direction
 * map, and write different planes, so nothing orders them). `batch` sets of
 * 1024 samples per workgroup. */
__global__ __launch_bounds__(256) void k_cdef(BatchDev B, int batch) {
  const AV1H_CMEM int32_t* pre_l = kernel_prefix(B, kKCdefLuma);
  const AV1H_CMEM int32_t* pre_c = kernel_prefix(B, kKCdefChroma);
  const int tl = pre_l[B.njobs], total = tl + pre_c[B.njobs];
  for (int base = 0; base < total; base += gridDim.x) {
    const int v = xcd_group(base, total);
    if (v < 0) continue;
    const bool luma = v < tl;
    const AV1H_CMEM int32_t* pre = luma ? pre_l : pre_c;
    const int vk = luma ? v : v - tl;
    const int j = find_job(pre, B.njobs, vk);
    FArgs a = filter_args(B, j);
    const int nl = a.plan.n_cdef_luma;
    for (int u = 0; u < batch; ++u)
      cdef_lane(a, luma ? 0 : nl, luma ? nl : a.plan.n_cdef - nl, (vk - pre[j]) * batch + u, luma);
  }
}

/* ---- superres (av1gpu_kernels.h:2387-2402) ------------------------------ */

typedef short lr_s2 __attribute__((ext_vector_type(2)));
/* two 16-bit products added to acc */
__device__ __forceinline__ int dot2(uint32_t a, uint32_t b, int acc) {
  return __builtin_amdgcn_sdot2(__builtin_bit_cast(lr_s2, a), __builtin_bit_cast(lr_s2, b), acc, false);
}
__device__ __forceinline__ uint32_t pack2(int lo, int hi) { return (uint32_t)(lo & 0xffff) | ((uint32_t)hi << 16); }

/* 256 x 16 output samples of one plane of one picture per workgroup, four
 * neighbouring samples of a row per lane: the source span of the 256 columns
 * (at most 264 samples when upscaling) is staged in LDS per row, eight bytes a
 * load, clamped to the coded width as each tap is (av1gpu_kernels.h:2387-2402).
 * A lane's columns stay the same down the rows, so their packed filters and
 * the shifts that align their taps are set up once. Picture 0 is the frame
 * (from the CDEF output in `scratch`; also stored to lr_cdef when loop
 * restoration reads it), picture 1 the deblocked picture loop restoration
 * reads (lr_curr into lr_prev_up). One sample per lane and row with 32-bit
 * products took 18 us on a 1080p frame, 57 on a 2160p one; now 12 and 30. */
constexpr int kUpW = 256, kUpRows = 16, kUpSpan = 280; /* from 3 to 6 samples left of the first tap's column */

/* output tiles of a plane of ow x oh display samples */
__host__ __device__ __forceinline__ int up_tiles(int ow, int oh) {
  return (ow + kUpW - 1) / kUpW * ((oh + kUpRows - 1) / kUpRows);
}

__device__ void upscale_tile(FArgs a, int t, const uint4* s_k, uint16_t (*s_row)[kUpSpan]) {
  LayRef L = a.lay;
  const int t0 = up_tiles(L.out_w[0], L.out_h[0]), t1 = up_tiles(L.out_w[1], L.out_h[1]);
  const int tp = t0 + t1 + up_tiles(L.out_w[2], L.out_h[2]);
  const int pic = t >= tp;
  int rem = t - pic * tp, p = 0;
  if (rem >= t0) {
    rem -= t0;
    p = 1;
    if (rem >= t1) {
      rem -= t1;
      p = 2;
    }
  }
  const int ow = L.out_w[p], oh = L.out_h[p];
  const int tx = (ow + kUpW - 1) / kUpW;
  const int by = rem / tx, bx = rem - by * tx;
  const uint16_t* src = (pic ? a.lr_curr : a.scratch) + L.plane_off[p];
  uint16_t* dst = (pic ? a.lr_prev_up : a.frame) + L.plane_off[p];
  uint16_t* dst2 = pic || !a.up_dst2 ? nullptr : a.up_dst2 + L.plane_off[p];
  const int x0 = bx * kUpW, y0 = by * kUpRows;
  const int step = a.up_step[p], init = a.up_initial[p];
  const int maxx = L.plane_w[p] - 1;
  const int stride = L.stride[p];
  const int xl = min(x0 + kUpW, ow) - 1;
  /* the first tap's column, down to a multiple of 4 */
  const int ws = (((-(1 << 14) + init + x0 * step) >> 14) - 3) & ~3;
  const int wn = ((-(1 << 14) + init + xl * step) >> 14) + 4 - ws + 1;
  const int rows = min(kUpRows, oh - y0);
  {
    /* all of a thread's loads issued before its LDS writes */
    constexpr int kQuads = kUpSpan / 4, kIt = (kQuads * kUpRows + 255) / 256;
    uint2 val[kIt];
#pragma unroll
    for (int u = 0; u < kIt; ++u) {
      const int e = (int)threadIdx.x + 256 * u, r = e / kQuads, c = 4 * (e - r * kQuads), x = ws + c;
      val[u] = make_uint2(0, 0);
      if (r >= rows || c >= wn) continue;
      const uint16_t* q = src + (size_t)(y0 + r) * stride;
      if (x >= 0 && x + 3 <= maxx) {
        val[u] = *reinterpret_cast<const uint2*>(q + x);
      } else {
        val[u].x = pack2(q[clampi(x, 0, maxx)], q[clampi(x + 1, 0, maxx)]);
        val[u].y = pack2(q[clampi(x + 2, 0, maxx)], q[clampi(x + 3, 0, maxx)]);
      }
    }
#pragma unroll
    for (int u = 0; u < kIt; ++u) {
      const int e = (int)threadIdx.x + 256 * u, r = e / kQuads;
      if (r < kUpRows) *reinterpret_cast<uint2*>(&s_row[r][4 * (e - r * kQuads)]) = val[u];
    }
  }
  __syncthreads();
  const int x = x0 + 4 * ((int)threadIdx.x & 63), n = xl - x + 1;
  if (n <= 0) return;
  uint4 k[4];
  int word[4], sh[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int sx = -(1 << 14) + init + min(x + i, xl) * step;
    const int o = (sx >> 14) - 3 - ws;
    k[i] = s_k[(sx & ((1 << 14) - 1)) >> 8];
    word[i] = o >> 1;
    sh[i] = (o & 1) * 16;
  }
  for (int r = (int)threadIdx.x >> 6; r < rows; r += 4) {
    int v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t* w = reinterpret_cast<const uint32_t*>(s_row[r]) + word[i];
      uint32_t m[5];
#pragma unroll
      for (int q = 0; q < 5; ++q) m[q] = w[q];
#pragma unroll
      for (int q = 0; q < 4; ++q) m[q] = __builtin_amdgcn_alignbit(m[q + 1], m[q], sh[i]);
      v[i] = clampi(dot2(m[3], k[i].w, dot2(m[2], k[i].z, dot2(m[1], k[i].y, dot2(m[0], k[i].x, 64)))) >> 7, 0, a.maxv);
    }
    const size_t at = (size_t)(y0 + r) * stride + x;
    if (n >= 4) {
      const uint2 w = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
      *reinterpret_cast<uint2*>(dst + at) = w;
      if (dst2) *reinterpret_cast<uint2*>(dst2 + at) = w;
    } else {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (i < n) {
          dst[at + i] = (uint16_t)v[i];
          if (dst2) dst2[at + i] = (uint16_t)v[i];
        }
    }
  }
}

__global__ __launch_bounds__(256) void k_upscale(BatchDev B) {
  __shared__ uint4 s_k[64]; /* a phase's eight taps, two a word */
  __shared__ __align__(16) uint16_t s_row[kUpRows][kUpSpan];
  {
    const int* q = &av1t_spec_table[AV1T_OFF_UPSCALE + 2 * threadIdx.x];
    reinterpret_cast<uint32_t*>(s_k)[threadIdx.x] = pack2(q[0], q[1]);
  }
  __syncthreads();
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKUpscale);
  const int total = pre[B.njobs];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int j = find_job(pre, B.njobs, v);
    upscale_tile(filter_args(B, j), v - pre[j], s_k, s_row);
    __syncthreads();
  }
}

/* ---- loop restoration (av1gpu_kernels.h:2832-2982) ---------------------- */

/* a2 of the self-guided filter for z = 0 .. 255 (the specification's
 * x_by_xplus1 mapping, av1gpu_kernels.h:2898): z >= 255 gives 256 */
__device__ __forceinline__ int sgr_a2(int z) { return z == 0 ? 1 : ((z << 8) + z / 2) / (z + 1); }

/* Loop restoration of one tile (at most kLrTileCols x kLrTileRows samples of
 * one restoration job, i.e. one unit inside one 64 row stripe) per workgroup,
 * four neighbouring samples per lane:
 *   the source window with its halo is staged in LDS as 16-bit samples,
 *   through the stripe rule (rows above / below the stripe from the deblocked
 *   picture, at most two away), eight bytes a load inside the picture;
 *   Wiener - the horizontal 7 tap pass into a 16-bit LDS intermediate (rounded
 *            and clamped to 15 bits and a sign), then the vertical pass
 *            (av1gpu_kernels.h:2832-2870), taps two at a time;
 *   SGR    - a lane walks a column of six positions down with its 5 and 3 wide
 *            row sums in registers; A and B of both passes, packed in a word
 *            (A at most 256; B at most 255 * 25 * 4095 * 164 >> 12 < 2^20), at
 *            every position the 3x3 neighbourhoods of the tile touch, pass 0
 *            only on the odd rows it weighs; then the weighted neighbourhood
 *            sums and the projection (av1gpu_kernels.h:2872-2982).
 * Bound by instructions: one sample per lane with 32-bit LDS samples and
 * multiplies took 37 us on a 1080p frame, 133 on a 2160p one, 50 on eight
 * streams (Wiener); now 19, 61 and 38, with a 64 x 16 tile in 13.6 KB. */
constexpr int kLrW = kLrTileCols, kLrH = kLrTileRows;
constexpr int kLrSrcLd = kLrW + 12, kLrSrcRows = kLrH + 6; /* from 4 left, 3 above */
constexpr int kLrMidLd = kLrW + 4, kLrAbLd = kLrW + 4, kLrAbRows = kLrH + 2;

struct LrLds {
  __align__(16) uint16_t src[kLrSrcRows * kLrSrcLd];
  union {
    __align__(16) int16_t mid[kLrSrcRows * kLrMidLd]; /* Wiener */
    __align__(16) uint32_t ab[2][kLrAbRows * kLrAbLd]; /* SGR, B << 9 | A */
  };
  uint16_t a2[256];
};

__device__ __forceinline__ void lr_store(uint16_t* dst, const int* v, int n, bool aligned) {
  if (n >= 4 && aligned) {
    uint2 w;
    w.x = pack2(v[0], v[1]);
    w.y = pack2(v[2], v[3]);
    *reinterpret_cast<uint2*>(dst) = w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n) dst[i] = (uint16_t)v[i];
  }
}

__device__ __forceinline__ void lr_wiener(LrLds& S, const DevLr& j, int bd, int maxv, int tw, int th, uint16_t* dst,
                                          int stride, bool aligned) {
  const int r0 = bd == 12 ? 5 : 3, r1 = bd == 12 ? 9 : 11;
  const int off = 1 << (bd + 7 - r0 - 1);
  const int top = (1 << (bd + 1 + 7 - r0)) - 1 - off;
  int ht[7], vt[7];
  bool narrow = true;
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    vt[t] = vt[6 - t] = j.vf[t];
    ht[t] = ht[6 - t] = j.hf[t];
  }
  vt[3] = 128 - 2 * (j.vf[0] + j.vf[1] + j.vf[2]);
  ht[3] = 128 - 2 * (j.hf[0] + j.hf[1] + j.hf[2]);
#pragma unroll
  for (int t = 0; t < 4; ++t)
    narrow = narrow && abs(ht[t]) < 8192 && abs(vt[t]) < 8192;
  const int quads = (tw + 3) >> 2, k = threadIdx.x & 15;
  if (!narrow) {
    /* taps beyond 13 bits and a sign (no stream codes them), whose sums of
     * products could leave 32 bits: one product at a time */
    for (int r = threadIdx.x >> 4; r < th + 6; r += 16)
      for (int i = 0; k < quads && i < 4; ++i) {
        int sum = 0;
        for (int t = 0; t < 7; ++t) sum += ht[t] * (int)S.src[r * kLrSrcLd + 4 * k + i + 1 + t];
        S.mid[r * kLrMidLd + 4 * k + i] = (int16_t)clampi(rsr64(sum, r0), -off, top);
      }
    __syncthreads();
    for (int r = threadIdx.x >> 4; r < th; r += 16)
      for (int i = 0; k < quads && i < 4 && 4 * k + i < tw; ++i) {
        int sum = 0;
        for (int t = 0; t < 7; ++t) sum += vt[t] * (int)S.mid[(r + t) * kLrMidLd + 4 * k + i];
        dst[(size_t)r * stride + 4 * k + i] = (uint16_t)clampi(rsr64(sum, r1), 0, maxv);
      }
    return;
  }
  const uint32_t h01 = pack2(ht[0], ht[1]), h23 = pack2(ht[2], ht[3]), h45 = pack2(ht[4], ht[5]), h6 = pack2(ht[6], 0);
  for (int r = threadIdx.x >> 4; r < th + 6; r += 16) {
    if (k >= quads) break;
    /* samples x - 4 .. x + 7 */
    const uint2* q = reinterpret_cast<const uint2*>(S.src + r * kLrSrcLd + 4 * k);
    const uint2 q0 = q[0], q1 = q[1], q2 = q[2];
    const uint32_t w[6] = {q0.x, q0.y, q1.x, q1.y, q2.x, q2.y};
    uint32_t m[5];
#pragma unroll
    for (int t = 0; t < 5; ++t) m[t] = __builtin_amdgcn_alignbit(w[t + 1], w[t], 16);
    const int half = 1 << (r0 - 1);
    int v[4];
    v[0] = dot2(m[3], h6, dot2(m[2], h45, dot2(m[1], h23, dot2(m[0], h01, half))));
    v[1] = dot2(w[4], h6, dot2(w[3], h45, dot2(w[2], h23, dot2(w[1], h01, half))));
    v[2] = dot2(m[4], h6, dot2(m[3], h45, dot2(m[2], h23, dot2(m[1], h01, half))));
    v[3] = dot2(w[5], h6, dot2(w[4], h45, dot2(w[3], h23, dot2(w[2], h01, half))));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = clampi(v[i] >> r0, -off, top);
    uint2 out;
    out.x = pack2(v[0], v[1]);
    out.y = pack2(v[2], v[3]);
    *reinterpret_cast<uint2*>(S.mid + r * kLrMidLd + 4 * k) = out;
  }
  __syncthreads();
  const uint32_t v01 = pack2(vt[0], vt[1]), v23 = pack2(vt[2], vt[3]), v45 = pack2(vt[4], vt[5]), v6 = pack2(vt[6], 0),
                 v6h = pack2(0, vt[6]);
  const int r = threadIdx.x >> 4;
  if (r < th && k < quads) {
    const int half = 1 << (r1 - 1);
    int v[4] = {half, half, half, half};
    const uint32_t vv[3] = {v01, v23, v45};
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const uint2 u = *reinterpret_cast<const uint2*>(S.mid + (r + 2 * t) * kLrMidLd + 4 * k);
      const uint2 d = *reinterpret_cast<const uint2*>(S.mid + (r + 2 * t + 1) * kLrMidLd + 4 * k);
      v[0] = dot2(__builtin_amdgcn_perm(d.x, u.x, 0x05040100u), vv[t], v[0]);
      v[1] = dot2(__builtin_amdgcn_perm(d.x, u.x, 0x07060302u), vv[t], v[1]);
      v[2] = dot2(__builtin_amdgcn_perm(d.y, u.y, 0x05040100u), vv[t], v[2]);
      v[3] = dot2(__builtin_amdgcn_perm(d.y, u.y, 0x07060302u), vv[t], v[3]);
    }
    const uint2 e = *reinterpret_cast<const uint2*>(S.mid + (r + 6) * kLrMidLd + 4 * k);
    v[0] = dot2(e.x, v6, v[0]);
    v[1] = dot2(e.x, v6h, v[1]);
    v[2] = dot2(e.y, v6, v[2]);
    v[3] = dot2(e.y, v6h, v[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = clampi(v[i] >> r1, 0, maxv);
    lr_store(dst + (size_t)r * stride + 4 * k, v, tw - 4 * k, aligned);
  }
}

/* A and B of one position of a pass from its box sums (at most 25 samples of
 * 12 bits), n samples in the box */
__device__ __forceinline__ uint32_t sgr_ab(int sq, int sum, int n, uint32_t mt, uint32_t inv, int bd, const uint16_t* a2s) {
  int sa = sq, sb = sum;
  if (bd > 8) {
    sa = rnd2(sa, 2 * (bd - 8));
    sb = rnd2(sb, bd - 8);
  }
  const int pp = max(0, sa * n - sb * sb);
  const uint32_t z = (uint32_t)(((uint64_t)(uint32_t)pp * mt + (1u << 19)) >> 20);
  const uint32_t a2 = z >= 255 ? 256 : a2s[z];
  const uint32_t b = ((256 - a2) * (uint32_t)sum * inv + (1u << 11)) >> 12;
  return b << 9 | a2;
}

__device__ __forceinline__ void lr_sgr(LrLds& S, const DevLr& j, int bd, int maxv, int tw, int th, int y0, uint16_t* dst,
                                       int stride, bool aligned) {
  constexpr int kQ = kLrW + 2, kRun = 6; /* columns of positions, rows a lane walks */
  static_assert(kQ * (kLrAbRows / kRun) <= 256 && kLrAbRows % kRun == 0, "self-guided positions per lane");
  const bool p0 = j.r[0] != 0, p1 = j.r[1] != 0;
  const int q = threadIdx.x % kQ, g = threadIdx.x / kQ;
  if (g < kLrAbRows / kRun && q < tw + 2) {
    uint32_t mt[2], inv[2];
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
      const int n = pass ? 9 : 25;
      const uint32_t n2e = (uint32_t)(n * n) * (uint32_t)max(j.eps[pass], 1);
      mt[pass] = ((1u << 20) + n2e / 2) / n2e;
      inv[pass] = ((1 << 12) + n / 2) / n;
    }
    /* row sums of the walked rows: five wide, three wide, and of squares */
    int h5[kRun + 4], s5[kRun + 4], h3[kRun + 4], s3[kRun + 4];
    const int sh = ((q + 1) & 1) * 16;
    const uint32_t* col = reinterpret_cast<const uint32_t*>(S.src + kRun * g * kLrSrcLd + ((q + 1) & ~1));
#pragma unroll
    for (int i = 0; i < kRun + 4; ++i) {
      const uint32_t w0 = col[i * (kLrSrcLd / 2)], w1 = col[i * (kLrSrcLd / 2) + 1], w2 = col[i * (kLrSrcLd / 2) + 2];
      const uint32_t a = __builtin_amdgcn_alignbit(w1, w0, sh), b = __builtin_amdgcn_alignbit(w2, w1, sh),
                     c = (w2 >> sh) & 0xffffu;
      const int first = (int)(a & 0xffffu), last = (int)c;
      const int mh = dot2(b, 0x00010001u, (int)(a >> 16));
      const int ms = dot2(b, b, __mul24((int)(a >> 16), (int)(a >> 16)));
      h3[i] = mh;
      s3[i] = ms;
      h5[i] = mh + first + last;
      s5[i] = ms + __mul24(first, first) + __mul24(last, last);
    }
    uint32_t* ab0 = S.ab[0] + kRun * g * kLrAbLd + q;
    uint32_t* ab1 = S.ab[1] + kRun * g * kLrAbLd + q;
    const int odd = (y0 - 1) & 1; /* kRun is even: of the run's first row */
#pragma unroll
    for (int i = 0; i < kRun; ++i) {
      if (p0 && ((i & 1) ^ odd))
        ab0[i * kLrAbLd] = sgr_ab(s5[i] + s5[i + 1] + s5[i + 2] + s5[i + 3] + s5[i + 4],
                                  h5[i] + h5[i + 1] + h5[i + 2] + h5[i + 3] + h5[i + 4], 25, mt[0], inv[0], bd, S.a2);
      if (p1)
        ab1[i * kLrAbLd] = sgr_ab(s3[i + 1] + s3[i + 2] + s3[i + 3], h3[i + 1] + h3[i + 2] + h3[i + 3], 9, mt[1], inv[1],
                                  bd, S.a2);
    }
  }
  __syncthreads();
  const int r = threadIdx.x >> 4, k = threadIdx.x & 15;
  if (r >= th || 4 * k >= tw) return;
  const int y = y0 + r;
  auto row = [&](int pass, int rr, uint32_t* v) {
    const uint32_t* p = S.ab[pass] + rr * kLrAbLd + 4 * k;
    const uint4 lo = *reinterpret_cast<const uint4*>(p);
    const uint2 hi = *reinterpret_cast<const uint2*>(p + 4);
    v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y;
  };
  const uint2 us = *reinterpret_cast<const uint2*>(S.src + (r + 3) * kLrSrcLd + 4 * k + 4);
  const int u[4] = {(int)(us.x & 0xffff), (int)(us.x >> 16), (int)(us.y & 0xffff), (int)(us.y >> 16)};
  int f0[4], f1[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) f0[i] = f1[i] = u[i] << 4;
  if (p0) {
    /* the odd rows among y - 1 .. y + 1, 5 6 5 across */
    uint32_t a[6], b[6], v[6];
    if (y & 1) {
      row(0, r + 1, v);
#pragma unroll
      for (int i = 0; i < 6; ++i) a[i] = v[i] & 511, b[i] = v[i] >> 9;
    } else {
      uint32_t d[6];
      row(0, r, v);
      row(0, r + 2, d);
#pragma unroll
      for (int i = 0; i < 6; ++i) a[i] = (v[i] & 511) + (d[i] & 511), b[i] = (v[i] >> 9) + (d[i] >> 9);
    }
    const int sh = 4 + ((y & 1) ? 4 : 5);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int sa = 5 * (int)(a[i] + a[i + 1] + a[i + 2]) + (int)a[i + 1];
      const int sb = 5 * (int)(b[i] + b[i + 1] + b[i + 2]) + (int)b[i + 1];
      f0[i] = rnd2(__mul24(sa, u[i]) + sb, sh);
    }
  }
  if (p1) {
    /* 3x3, 4 on the cross, 3 in the corners */
    uint32_t t[6], m[6], d[6];
    row(1, r, t);
    row(1, r + 1, m);
    row(1, r + 2, d);
    int ap[6], aq[6], bp[6], bq[6]; /* a column in the middle, at a side */
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const int ea = (int)((t[i] & 511) + (d[i] & 511)), eb = (int)((t[i] >> 9) + (d[i] >> 9));
      ap[i] = (ea + (int)(m[i] & 511)) << 2;
      bp[i] = (eb + (int)(m[i] >> 9)) << 2;
      aq[i] = ap[i] - ea;
      bq[i] = bp[i] - eb;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int sa = aq[i] + ap[i + 1] + aq[i + 2], sb = bq[i] + bp[i + 1] + bq[i + 2];
      f1[i] = rnd2(__mul24(sa, u[i]) + sb, 9);
    }
  }
  const int w0 = j.xqd[0], w1 = j.xqd[1], w2 = (1 << 7) - w0 - w1;
  int out[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int64_t v = (int64_t)w1 * (u[i] << 4);
    v += (int64_t)w0 * f0[i];
    v += (int64_t)w2 * f1[i];
    out[i] = clampi(rsr64(v, 4 + 7), 0, maxv);
  }
  lr_store(dst + (size_t)r * stride + 4 * k, out, tw - 4 * k, aligned);
}

__device__ __forceinline__ void lr_tile(FArgs a, int t, LrLds& S) {
  const int2 tile = a.plan.lr_tiles[t];
  const DevLr& j = a.plan.lr[tile.x];
  const int x0 = j.x + (tile.y & 0xffff), y0 = j.y + (tile.y >> 16);
  const int tw = min(kLrW, j.x + j.w - x0), th = min(kLrH, j.y + j.h - y0);
  LayRef L = a.lay;
  const int p = j.plane, bd = L.bit_depth;
  const int stride = L.stride[p], pw = L.out_w[p], ph = L.out_h[p], s0 = j.stripe0, s1 = j.stripe1;
  const uint16_t* cdef = a.lr_cdef + L.plane_off[p];
  const uint16_t* curr = (a.upscaled ? a.lr_prev_up : a.lr_curr) + L.plane_off[p];
  const bool aligned = (x0 & 3) == 0; /* units are multiples of 4 wide but for the smallest sizes */
  {
    /* all of a thread's loads issued before its LDS writes */
    constexpr int kQuads = kLrSrcLd / 4 - 1, kIt = (kQuads * kLrSrcRows + 255) / 256; /* columns -4 .. kLrW + 3 */
    uint2 val[kIt];
#pragma unroll
    for (int u = 0; u < kIt; ++u) {
      const int e = (int)threadIdx.x + 256 * u, r = e / kQuads, x = x0 - 4 + 4 * (e - r * kQuads);
      val[u] = make_uint2(0, 0);
      if (r >= th + 6 || x >= x0 + tw + 3) continue;
      const int y = clampi(y0 - 3 + r, 0, ph - 1);
      const uint16_t* src = y < s0 ? curr + (size_t)max(y, s0 - 2) * stride
                                   : y > s1 ? curr + (size_t)min(y, s1 + 2) * stride : cdef + (size_t)y * stride;
      if (aligned && x >= 0 && x + 3 < pw) {
        val[u] = *reinterpret_cast<const uint2*>(src + x);
      } else {
        val[u].x = pack2(src[clampi(x, 0, pw - 1)], src[clampi(x + 1, 0, pw - 1)]);
        val[u].y = pack2(src[clampi(x + 2, 0, pw - 1)], src[clampi(x + 3, 0, pw - 1)]);
      }
    }
#pragma unroll
    for (int u = 0; u < kIt; ++u) {
      const int e = (int)threadIdx.x + 256 * u, r = e / kQuads;
      if (r < kLrSrcRows) *reinterpret_cast<uint2*>(S.src + r * kLrSrcLd + 4 * (e - r * kQuads)) = val[u];
    }
  }
  __syncthreads();
  uint16_t* dst = a.frame + L.plane_off[p] + (size_t)y0 * stride + x0;
  if (j.type == 1)
    lr_wiener(S, j, bd, a.maxv, tw, th, dst, stride, aligned);
  else
    lr_sgr(S, j, bd, a.maxv, tw, th, y0, dst, stride, aligned);
}

__global__ __launch_bounds__(256) void k_lr(BatchDev B) {
  __shared__ LrLds S;
  S.a2[threadIdx.x] = (uint16_t)sgr_a2(threadIdx.x);
  __syncthreads();
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKLr);
  const int total = pre[B.njobs];
  for (int base = 0; base < total; base += gridDim.x) {
    const int v = xcd_group(base, total);
    if (v < 0) continue;
    const int j = find_job(pre, B.njobs, v);
    lr_tile(filter_args(B, j), v - pre[j], S);
    __syncthreads();
  }
}

/* ---- whole picture copies (the snapshots the filters read, the reference
 * slot store) ---------------------------------------------------------------- */

__device__ __forceinline__ void copy_kind(FArgs a, int k, const uint4** src, uint4** dst) {
  *src = reinterpret_cast<const uint4*>(a.frame);
  switch (k) {
    case kKCopyLrCurr: *dst = reinterpret_cast<uint4*>(a.lr_curr); break;
    case kKCopyCdefSrc:
    case kKCopyUpSrc: *dst = reinterpret_cast<uint4*>(a.scratch); break;
    default: *dst = reinterpret_cast<uint4*>(a.store); break;
  }
}

/* kCopyChunk bytes per workgroup, 16 bytes per thread and step */
__global__ __launch_bounds__(256) void k_copy(BatchDev B, int k) {
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, k);
  const int total = pre[B.njobs];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int j = find_job(pre, B.njobs, v);
    FArgs a = filter_args(B, j);
    const uint4* src;
    uint4* dst;
    copy_kind(a, k, &src, &dst);
    /* the deblocked snapshot may have a second destination */
    uint4* dst2 = k == kKCopyLrCurr ? reinterpret_cast<uint4*>(a.snap2) : nullptr;
    const int64_t n = a.lay.size * 2 / 16;
    const int64_t base = (int64_t)(v - pre[j]) * (kCopyChunk / 16);
#pragma unroll
    for (int i = 0; i < kCopyChunk / 16 / 256; ++i) {
      const int64_t e = base + i * 256 + threadIdx.x;
      if (e < n) {
        const uint4 x = src[e];
        dst[e] = x;
        if (dst2) dst2[e] = x;
      }
    }
  }
}

/* ---- NV12 and RGB packs (av1gpu_kernels.h:3379-3472) -------------------- */

/* one thread per output byte pair */
__global__ void k_nv12(Layout L, const uint16_t* src, uint8_t* out, int pitch) {
  const int x2 = (blockIdx.x * blockDim.x + threadIdx.x) * 2;
  const int row = blockIdx.y;
  if (x2 >= pitch) return;
  const int sh = L.bit_depth - 8;
  const int w = L.width, h = L.height;
  uint8_t* d = out + (size_t)row * pitch + x2;
  if (row < h) {
    const uint16_t* s = src + L.plane_off[0] + (size_t)row * L.stride[0];
    d[0] = x2 < w ? (uint8_t)(s[x2] >> sh) : 0;
    if (x2 + 1 < pitch) d[1] = x2 + 1 < w ? (uint8_t)(s[x2 + 1] >> sh) : 0;
    return;
  }
  const int cr = row - h;
  const int cw = (w + (1 << L.ss_x) - 1) >> L.ss_x;
  const int c = x2 >> 1;
  if (c < cw) {
    d[0] = (uint8_t)(src[L.plane_off[1] + (size_t)cr * L.stride[1] + c] >> sh);
    d[1] = (uint8_t)(src[L.plane_off[2] + (size_t)cr * L.stride[2] + c] >> sh);
  } else {
    d[0] = 0;
    if (x2 + 1 < pitch) d[1] = 0;
  }
}

/* NV12 of each frame of a batch that asks for it, after film grain: 1024
 * output bytes of one row per workgroup, 4 per thread */
__device__ void nv12_chunk(FArgs a, int t) {
  LayRef L = a.lay;
  const int pitch = a.nv12_pitch;
  const int cpr = (pitch + 1023) >> 10;
  const int row = t / cpr;
  const int x0 = (t - row * cpr) * 1024 + threadIdx.x * 4;
  if (x0 >= pitch) return;
  const int sh = L.bit_depth - 8, w = L.width, h = L.height;
  uint32_t word = 0;
  if (row < h) {
    const uint16_t* src = a.frame + L.plane_off[0] + (size_t)row * L.stride[0];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (x0 + k < w) word |= (uint32_t)(src[x0 + k] >> sh) << (8 * k);
  } else {
    const int cr = row - h, cw = (w + (1 << L.ss_x) - 1) >> L.ss_x;
    const uint16_t* u = a.frame + L.plane_off[1] + (size_t)cr * L.stride[1];
    const uint16_t* v = a.frame + L.plane_off[2] + (size_t)cr * L.stride[2];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int c = (x0 + k) >> 1;
      if (c < cw) word |= (uint32_t)(((x0 + k) & 1 ? v[c] : u[c]) >> sh) << (8 * k);
    }
  }
  uint8_t* d = a.nv12 + (size_t)row * pitch + x0;
  if ((pitch & 3) == 0 && x0 + 4 <= pitch) {
    *reinterpret_cast<uint32_t*>(d) = word;
  } else {
    for (int k = 0; k < 4 && x0 + k < pitch; ++k) d[k] = (uint8_t)(word >> (8 * k));
  }
}

__global__ __launch_bounds__(256) void k_nv12_batch(BatchDev B) {
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKNv12);
  const int total = pre[B.njobs];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int j = find_job(pre, B.njobs, v);
    nv12_chunk(filter_args(B, j), v - pre[j]);
  }
}

/* Picture checksums (mix64 weights, see the header): kHashChunk samples per
 * workgroup, 16 per thread, a wave sum added to the frame's accumulator. */
__global__ __launch_bounds__(256) void k_hash(BatchDev B) {
  const AV1H_CMEM int32_t* pre = kernel_prefix(B, kKHash);
  const int total = pre[B.njobs];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int j = find_job(pre, B.njobs, v);
    FArgs a = filter_args(B, j);
    LayRef L = a.lay;
    const int64_t n0 = (int64_t)L.out_w[0] * L.out_h[0], n1 = (int64_t)L.out_w[1] * L.out_h[1];
    const int64_t n = n0 + 2 * n1;
    uint64_t acc = 0;
    const int64_t base = (int64_t)(v - pre[j]) * kHashChunk;
#pragma unroll 4
    for (int k = 0; k < kHashChunk / 256; ++k) {
      const int64_t i = base + k * 256 + threadIdx.x;
      if (i < n) {
        int p = 0;
        int64_t r = i;
        if (r >= n0) {
          r -= n0;
          p = 1;
          if (r >= n1) {
            r -= n1;
            p = 2;
          }
        }
        const int w = L.out_w[p];
        const int y = (int)(r / w), x = (int)(r - (int64_t)y * w);
        acc += (uint64_t)a.frame[L.plane_off[p] + (int64_t)y * L.stride[p] + x] * mix64((uint64_t)i);
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if ((threadIdx.x & 63) == 0) atomicAdd((unsigned long long*)a.hash, (unsigned long long)acc);
  }
}

__global__ void k_zero64(uint64_t* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

/* The batch table (jobs, kernel prefixes, merged queue) copied from its
 * pinned staging buffer into device memory as the batch's first launch: the
 * byte count is the staging buffer's first word and the table follows at
 * kTableHead, so one captured launch serves every table size, and no copy
 * command of its own sits between two batches on the stream. The host
 * rewrites the staging buffer between the batches that use it: the loads
 * are system scope, past the device's caches. */
__global__ void k_fetch_table(const uint64_t* src, uint64_t* dst) {
  const uint64_t words = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) >> 3;
  const uint64_t* from = src + kTableHead / 8;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += 4 * stride) {
    uint64_t v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = i + k * stride < words ? __hip_atomic_load(from + i + k * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)
                                    : 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (i + k * stride < words) dst[i + k * stride] = v[k];
  }
}

/* The batch's results written into its pinned read-back buffer as its last
 * launch, instead of copies queued behind the batch: the error word (then
 * cleared for the next batch on the stream) and, with `hashes`, the n
 * pictures' checksums; system-scope stores, which the host reads once the
 * batch's completion event has fired. */
__global__ void k_readback(uint32_t* err, const uint64_t* hashes, int n, uint32_t* out_err, uint64_t* out_hash) {
  if (threadIdx.x == 0) {
    __hip_atomic_store(out_err, *err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    *err = 0;
  }
  if (hashes)
    for (int i = threadIdx.x; i < n; i += blockDim.x)
      __hip_atomic_store(out_hash + i, hashes[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct ColorM {
  int m[8];
  int o[3];
};

__global__ void k_rgb(Layout L, const uint16_t* src, uint8_t* out, ColorM cm) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y;
  if (x >= L.width) return;
  const int yy = src[L.plane_off[0] + (size_t)y * L.stride[0] + x];
  const size_t co = (size_t)(y >> L.ss_y) * L.stride[1] + (x >> L.ss_x);
  const int uu = src[L.plane_off[1] + co], vv = src[L.plane_off[2] + co];
  const int r = (cm.m[0] * yy + cm.m[1] * vv + cm.o[0]) >> 16;
  const int g = (cm.m[2] * yy + cm.m[3] * uu + cm.m[4] * vv + cm.o[1]) >> 16;
  const int b = (cm.m[5] * yy + cm.m[6] * uu + cm.o[2]) >> 16;
  uint8_t* d = out + ((size_t)y * L.width + x) * 3;
  d[0] = (uint8_t)clampi(r, 0, 255);
  d[1] = (uint8_t)clampi(g, 0, 255);
  d[2] = (uint8_t)clampi(b, 0, 255);
}

}  // namespace

void superres_params(int dw, int uw, int* step, int* initial) {
  /* av1gpu_kernels.h:2375-2383 */
  const int st = ((dw << 14) + (uw / 2)) / uw;
  const int err = uw * st - (dw << 14);
  const int sub = (-((uw - dw) << 13) + uw / 2) / uw + (1 << 7) - err / 2;
  *step = st;
  *initial = sub & ((1 << 14) - 1);
}

int upscale_tiles(const Layout& L, int pictures) {
  return (up_tiles(L.out_w[0], L.out_h[0]) + up_tiles(L.out_w[1], L.out_h[1]) + up_tiles(L.out_w[2], L.out_h[2])) *
         pictures;
}

hipError_t launch_filter_kernel(const BatchDev& b, int k, int total, int cap, int cdef_batch, hipStream_t s) {
  const dim3 blk(256), grid(min(total, cap));
  switch (k) {
    case kKDeblockV:
    case kKDeblockH: hipLaunchKernelGGL(k_deblock, grid, blk, 0, s, b, k == kKDeblockH ? 1 : 0); break;
    case kKCdefDir: hipLaunchKernelGGL(k_cdef_dir, grid, blk, 0, s, b); break;
    case kKCdefLuma:
      /* luma and chroma in one launch (kKCdefLuma's): `total` counts both */
      hipLaunchKernelGGL(k_cdef, grid, blk, 0, s, b, cdef_batch);
      break;
    case kKUpscale: hipLaunchKernelGGL(k_upscale, grid, blk, 0, s, b); break;
    case kKLr: hipLaunchKernelGGL(k_lr, grid, blk, 0, s, b); break;
    case kKNv12: hipLaunchKernelGGL(k_nv12_batch, grid, blk, 0, s, b); break;
    case kKHash: hipLaunchKernelGGL(k_hash, grid, blk, 0, s, b); break;
    case kKCopyLrCurr:
    case kKCopyCdefSrc:
    case kKCopyUpSrc:
    case kKCopyStore: hipLaunchKernelGGL(k_copy, grid, blk, 0, s, b, k); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_zero64(uint64_t* p, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_zero64, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t launch_fetch_table(const void* pin, void* dev, int frames, hipStream_t s) {
  /* a table the launch fetches is one frame's, a few KB */
  (void)frames;
  hipLaunchKernelGGL(k_fetch_table, dim3(1), dim3(256), 0, s, static_cast<const uint64_t*>(pin),
                     static_cast<uint64_t*>(dev));
  return hipGetLastError();
}

hipError_t launch_readback(uint32_t* err, const uint64_t* hashes, int n, uint32_t* out_err, uint64_t* out_hash,
                           hipStream_t s) {
  hipLaunchKernelGGL(k_readback, dim3(1), dim3(64), 0, s, err, hashes, n, out_err, out_hash);
  return hipGetLastError();
}

hipError_t launch_nv12(const Layout& lay, const uint16_t* src, uint8_t* out, int pitch, hipStream_t s) {
  const int rows = lay.height + ((lay.height + (1 << lay.ss_y) - 1) >> lay.ss_y);
  hipLaunchKernelGGL(k_nv12, dim3((pitch / 2 + 127) / 128, rows), dim3(128), 0, s, lay, src, out, pitch);
  return hipGetLastError();
}

hipError_t launch_rgb(const Layout& lay, const uint16_t* src, uint8_t* out, const int m[8], const int o[3],
                      hipStream_t s) {
  ColorM cm;
  for (int i = 0; i < 8; ++i) cm.m[i] = m[i];
  for (int i = 0; i < 3; ++i) cm.o[i] = o[i];
  hipLaunchKernelGGL(k_rgb, dim3((lay.width + 127) / 128, lay.height), dim3(128), 0, s, lay, src, out, cm);
  return hipGetLastError();
}

}  // namespace av1hip
