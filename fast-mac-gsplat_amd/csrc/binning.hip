// binning.hip -- per-splat tile-hit counts, record packing, deterministic
// (tile, gid) pair emission and tile-range extraction.
//
// This translation unit is compiled with -ffp-contract=off: the predicate
// results must match the CPU oracle bit for bit.
//
// Row walk (the count and emit kernels).  The candidate tiles of a splat are
// the tiles of its snug pixel bbox; a candidate is a hit when the tile's
// pixel-centre rectangle meets the splat's alpha >= threshold ellipse
// (reference count_tiles / emit_binned_ids,
// variants/v8/csrc/metal/gsplat_v8_kernels.metal:244-327).  A wavefront takes
// kWalkSplats (32) splats, prefix-sums the rows of their tile boxes and takes
// 64 rows per step whatever splats they belong to; each lane finds its row's
// span of hits from the ellipse (span_constants) and tests exactly only the
// tiles that the span's bounds leave open.  The walk is bound by the vector
// instructions it issues, and testing every candidate tile took them: a 3D
// scene's splats have 45 candidates in 7 rows.  The counts add up spans; the
// emits lay a step's spans end to end and write 64 pairs at a time.  Measured
// (us, every tile tested -> spans): two images of 100K 3D splats at 29 pairs
// each, count 61 -> 19, emit 69 -> 45; 200K at 40 pairs, count 78 -> 18, emit
// 82 -> 54 (from the count's recorded hits before); 64K 2D splats of 4.5
// pairs, count 11.9 -> 11.2, emit 13.1 -> 13.8.
//
// Staged path (one launch per step, also the separate C-ABI steps):
// count_kernel  original order: per-splat hit counts and per-workgroup sums
//   (sum_kernel turns them into the pair count N).
// pack_kernel   one thread per depth-sorted splat (gid): packed 64-byte
//   record and exclusive per-gid pair offsets (workgroup scan + decoupled
//   look-back in the same launch).
// emit_kernel   gid order: each hit claims a slot in its splat's range
//   [splat_offsets[gid], splat_offsets[gid+1]) and writes (tile, gid); the
//   same launch zeroes the pair sort's look-back status and counts the pair
//   sort's digit histograms per workgroup (reduced by hist_reduce_kernel).
//   Pairs of one splat have distinct tiles and splats occupy consecutive
//   ranges in gid order, so a stable sort by tile yields (tile, gid) order
//   whatever order the slots inside a splat's range were claimed in.
// ranges_kernel / counts_kernel  tile_offsets and tile_counts from the
//   sorted tile keys (the reference reads them from its atomic counters).
//
// Images of at most 131,072 splats whose pair count goes to host memory
// (the per-step path) take fewer launches:
// count_depth_runs_kernel  the count blocks above beside the depth sort's
//   run-sorting blocks, in one launch.
// rank_pack_kernel  the depth sort's rank step, packing each record where
//   its rank lands and adding each gid's hit count to the total of the emit
//   workgroup that holds the gid.
// emit_kernel<true>  scans its gids' counts from the sum of the totals of
//   the workgroups before it (no look-back), then emits as above.
// bucket_sort_kernel  after one onesweep pass on the high tile bits, a
//   counting sort of each bucket of 2^(bits-8) tiles on the low bits that
//   also writes the tile ranges (images of 2^9..2^16 tiles whose pair
//   buffer holds at most 4096 pairs per bucket on average).
// host_report_kernel  the binning's report to host memory where the
//   forward compositor does not write it.
//
// Larger images in one call: count_kernel also keeps the splats' records in
// original order; pack_kernel gives each original index its pair offset and
// gid; and emit_kernel<false, true> walks the splats in the count's original
// order.
#include <algorithm>

#include "gs_internal.h"
#include "gs_predicate.h"
#include "depth_runs.h"
#include "record.h"
#include "lookback.h"

namespace gs {
namespace {

constexpr int kThreads = 256;

struct SplatGeom {
  float mx, my, a, b, c, o;
};

constexpr int kWaves = kThreads / 64;

// Splats per wavefront in the row walk.  A wavefront's 64 lanes take the
// rows of kS splats together; fewer splats per wavefront
// than lanes gives each launch more wavefronts (the walk is latency bound)
// and a shorter slot search.  kS is kWalkSplats, or fewer in the small-image
// path where few splats have many candidates each (walk_splats).
constexpr int kWalkSplats = 32;
constexpr int kWalkBlockSplats = kWaves * kWalkSplats;
// Emit launches with at most this many workgroups add their pair-sort
// histograms atomically instead of through hist_reduce_kernel.
constexpr int kDirectHistBlocks = 1024;
// Copies of the emit's digit histograms (see emit_kernel).
constexpr int kHistCopies = 2;

// One wavefront's kS splats, staged for the cooperative row walk.
template <int kS>
struct WalkSlots {
  float4 g0[kS];   // mx, my, a, b
  float4 g1[kS];   // c, tau, kc, ka
  float4 span[kS]; // SpanConst
  int4 box[kS];    // tx0, ty0, tx1, first tile of the image
  float margin[kS];  // of the spans' ends (pixels); < 0: no certain spans
  int flags[kS];   // bit 0: use_c, bit 1: use_a
  int cend[kS];    // inclusive prefix sum of the boxes' rows
  int first[kS];   // exclusive prefix sum: the splat's first row
  uint32_t own[64];  // per walk step: items starting at each position
};

// Inclusive prefix maximum over the wavefront's 64 lanes (DPP: row shifts by
// 1, 2, 4, 8, then the row broadcasts carry rows 0 and 2 into rows 1, 3 and
// row 1 into rows 2, 3).  Lanes without a DPP source see 0, the identity.
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROW_MASK, 0xF,
                                               false);
}
__device__ __forceinline__ uint32_t wave_prefix_max(uint32_t x) {
  x = max(x, dpp_or_zero<0x111>(x));
  x = max(x, dpp_or_zero<0x112>(x));
  x = max(x, dpp_or_zero<0x114>(x));
  x = max(x, dpp_or_zero<0x118>(x));
  x = max(x, dpp_or_zero<0x142, 0xA>(x));
  x = max(x, dpp_or_zero<0x143, 0xC>(x));
  return x;
}

// Inclusive prefix sum over the wavefront's 64 lanes, the same way.
__device__ __forceinline__ int wave_prefix_sum(int v) {
  uint32_t x = (uint32_t)v;
  x += dpp_or_zero<0x111>(x);
  x += dpp_or_zero<0x112>(x);
  x += dpp_or_zero<0x114>(x);
  x += dpp_or_zero<0x118>(x);
  x += dpp_or_zero<0x142, 0xA>(x);
  x += dpp_or_zero<0x143, 0xC>(x);
  return (int)x;
}

// The rows of a splat's tile box hold its hits in one span each, and a row's
// span is found from the ellipse itself instead of testing every tile: for
// dy in the row's [dy0, dy1] the points with q(dx, dy) <= t reach to
//   dx = ka dy +- sqrt(t/a - (det/a^2) dy^2),  ka = -b/a,
// which is largest at the ellipse's rightmost point dy = kc hx (kc = -b/c,
// hx = sqrt(t c/det)), or at the end of the row next to it.  Evaluated for
// t = tau (1 + d) and t = tau (1 - d), d = 2^-10, this gives a span outside
// which no tile passes ellipse_hits_rect and one inside which every tile
// does; the tiles between the two (almost always none) are tested exactly.
//
// Why d suffices: the predicate's rounded quadratics (operands dx, dy of one
// rounded subtraction each, relative error 2^-24) differ from the exact ones
// by less than 16 2^-24 S, S = a dx^2 + c dy^2, and S <= q / (1 - r) with
// r^2 = b^2 / (a c).  Spans are used where 1 - r^2 = det / (a c) >= 2^-7, so
// 1 - r >= 2^-8 and the difference is below 2^-12 q.  A tile whose exact
// minimum is at most tau (1 - d) is thus found by the predicate (which
// evaluates each edge's own minimum, off by a rounded slope: second order),
// and one whose exact minimum is above tau (1 + d) has every evaluated term
// above tau.  det's own relative error, below 2^-22 2^7, moves t/a -
// (det/a^2) dy^2 by 2^-15 of t/a, far below d, and the clamped dy by an
// amount whose effect at the maximum is second order (below 2^-23 hx).  The
// rounding of mx + dx is covered by a margin of 2^-20 (|mx| + hx) + 2^-20.
// Rows of other splats (thin ones, c or a at most 1e-8, anything not finite)
// have no certain span: every tile is tested.
constexpr float kSpanUp = 1.0f + 0x1p-10f;
constexpr float kSpanDown = 1.0f - 0x1p-10f;

// {tau (1 + d) / a, tau (1 - d) / a, det / a^2, kc hx at tau (1 + d)}; margin
// < 0 where spans are not used.
__device__ __forceinline__ float4 span_constants(const SplatGeom& s, float tau,
                                                 const ConicSlopes& k,
                                                 float& margin) {
#pragma clang fp contract(off)
  margin = -1.0f;
  const float det = s.a * s.c - s.b * s.b;
  if (!(k.use_a && k.use_c && s.a < 0x1p60f && s.c < 0x1p60f &&
        det >= 0x1p-7f * (s.a * s.c) && fabsf(s.mx) < 0x1p30f &&
        fabsf(s.my) < 0x1p30f))
    return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float hx = __builtin_sqrtf(tau * kSpanUp * s.c / det);
  if (!(hx < 0x1p30f)) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  margin = (fabsf(s.mx) + hx) * 0x1p-20f + 0x1p-20f;
  return make_float4(tau * kSpanUp / s.a, tau * kSpanDown / s.a,
                     det / s.a / s.a, k.kc * hx);
}

// A row's tiles [m0, m1] that may hit and, of those, [c0, c1] that certainly
// do (c0 > m1 when none).
struct RowSpan {
  int m0, m1, c0, c1;
};

template <int kS>
__device__ __forceinline__ RowSpan row_span(const RasterParams& P,
                                            const WalkSlots<kS>& W, int sl,
                                            int ty) {
#pragma clang fp contract(off)
  const int4 bx = W.box[sl];
  const float margin = W.margin[sl];
  RowSpan r{bx.x, bx.z, 0x7fffffff, 0x7fffffff};
  if (margin < 0.0f) return r;
  const float4 g0 = W.g0[sl], sc = W.span[sl];
  const float ka = W.g1[sl].w;
  const float dy0 = (float)(ty * 16) + 0.5f - g0.y;
  const float dy1 =
      fminf((float)(P.height - 1) + 0.5f, (float)(ty * 16 + 15) + 0.5f) - g0.y;
  const float yr = fminf(fmaxf(sc.w, dy0), dy1);
  const float yl = fminf(fmaxf(-sc.w, dy0), dy1);
  const float dr = sc.x - sc.z * yr * yr, dl = sc.x - sc.z * yl * yl;
  const float lo = (float)bx.x, hi = (float)bx.z;
  if (dr < 0.0f || dl < 0.0f) {  // the row lies beyond the ellipse
    r.m1 = r.m0 - 1;
    return r;
  }
  const float xr = g0.x + (ka * yr + __builtin_amdgcn_sqrtf(dr));
  const float xl = g0.x + (ka * yl - __builtin_amdgcn_sqrtf(dl));
  // tiles t with 16 t + 0.5 <= xr and 16 t + 15.5 >= xl
  r.m0 = (int)fminf(fmaxf(ceilf((xl - margin - 15.5f) * 0.0625f), lo), hi + 1.0f);
  r.m1 = (int)fmaxf(fminf(floorf((xr + margin - 0.5f) * 0.0625f), hi), lo - 1.0f);
  const float inw = sc.w * kSpanDown;
  const float zr = fminf(fmaxf(inw, dy0), dy1);
  const float zl = fminf(fmaxf(-inw, dy0), dy1);
  const float er = sc.y - sc.z * zr * zr, el = sc.y - sc.z * zl * zl;
  if (er < 0.0f || el < 0.0f) return r;
  const float ur = g0.x + (ka * zr + __builtin_amdgcn_sqrtf(er));
  const float ul = g0.x + (ka * zl - __builtin_amdgcn_sqrtf(el)) + margin;
  const int c0 = (int)fminf(fmaxf(ceilf((ul - 15.5f) * 0.0625f), lo), hi + 1.0f);
  int c1 = (int)fmaxf(fminf(floorf((ur - margin - 0.5f) * 0.0625f), hi), lo - 1.0f);
  // (the image's last column of tiles may end before 16 t + 15.5)
  if (c1 == P.tiles_x - 1 && !((float)(P.width - 1) + 0.5f >= ul)) --c1;
  if (c0 <= c1 && c0 >= r.m0 && c1 <= r.m1) {
    r.c0 = c0;
    r.c1 = c1;
  }
  return r;
}

// The exact test of one tile of the slot's splat.
template <int kS>
__device__ __forceinline__ bool tile_hit(const RasterParams& P,
                                         const WalkSlots<kS>& W, int sl,
                                         int tx, int ty) {
  const float4 g0 = W.g0[sl], g1 = W.g1[sl];
  const int fl = W.flags[sl];
  ConicSlopes ks;
  ks.kc = g1.z;
  ks.ka = g1.w;
  ks.use_c = (fl & 1) != 0;
  ks.use_a = (fl & 2) != 0;
  float rx0, ry0, rx1, ry1;
  tile_rect(tx, ty, P.width, P.height, rx0, ry0, rx1, ry1);
  return ellipse_hits_rect(g0.x, g0.y, g0.z, g0.w, g1.x, ks, g1.y, rx0, ry0,
                           rx1, ry1);
}

// Stages this lane's splat (lanes below kS) and returns the rows of the
// wavefront's boxes.  With P.live the box is P.boxes[source], which holds
// the live tiles.  Rows fit in int32: tiles per image are limited to 2^24 on
// the host.
template <int kS>
__device__ __forceinline__ int walk_setup(const RasterParams& P, bool valid,
                                          const SplatGeom& s, int batch,
                                          int source, WalkSlots<kS>& W) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  int rows = 0;
  int4 box = make_int4(0, 0, -1, 0);
  float tau = 0.0f;
  if (valid && alpha_support(s.o, P.alpha_thr, P.eps, tau)) {
    if (P.live != nullptr) {
      const uint2 lb = P.boxes[source];
      if (lb.y != 0u) {
        box = make_int4((int)(lb.x & 0xffffu), (int)(lb.x >> 16),
                        (int)(lb.x & 0xffffu) + (int)(lb.y & 0xffffu) - 1,
                        batch * P.tiles_per_image);
        rows = (int)(lb.y >> 16);
      }
    } else {
      const PixBox bb =
          snugbox(s.mx, s.my, s.a, s.b, s.c, tau, P.width, P.height, P.eps);
      if (bb.x0 <= bb.x1 && bb.y0 <= bb.y1) {
        box = make_int4(bb.x0 >> 4, bb.y0 >> 4, bb.x1 >> 4,
                        batch * P.tiles_per_image);
        rows = (bb.y1 >> 4) - box.y + 1;
      }
    }
  }
  int inc = rows;
#pragma unroll
  for (int off = 1; off < kS; off <<= 1) {
    const int y = __shfl_up(inc, off, 64);
    if (lane >= off) inc += y;
  }
  if (lane < kS) {
    ConicSlopes k{0.0f, 0.0f, false, false};
    float margin = -1.0f;
    float4 span = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (rows > 0) {
      k = conic_slopes(s.a, s.b, s.c);
      span = span_constants(s, tau, k, margin);
    }
    W.g0[lane] = make_float4(s.mx, s.my, s.a, s.b);
    W.g1[lane] = make_float4(s.c, tau, k.kc, k.ka);
    W.span[lane] = span;
    W.box[lane] = box;
    W.margin[lane] = margin;
    W.flags[lane] = (k.use_c ? 1 : 0) | (k.use_a ? 2 : 0);
    W.cend[lane] = inc;
    W.first[lane] = inc - rows;
  }
  __builtin_amdgcn_wave_barrier();
  return __shfl(inc, kS - 1, 64);
}

// The lane whose items cover position base + lane, given every lane's first
// item (ascending; a lane without items shares its first with the next one
// and loses to it): the owner of position base is counted with a ballot, the
// lanes that start inside the 64 positions mark theirs with an LDS max, and a
// prefix maximum spreads the marks -- one LDS round trip instead of a binary
// search.
__device__ __forceinline__ int owner_lane(uint32_t* own, int first, int base) {
  const int lane = threadIdx.x & 63;
  const int owner0 = __popcll(__ballot(first <= base)) - 1;  // first[0] = 0
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  own[lane] = lane == 0 ? (uint32_t)owner0 : 0u;
  if (first > base && first < base + 64)
    atomicMax(&own[first - base], (uint32_t)lane);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return (int)wave_prefix_max(own[lane]);
}

// The wavefront's rows 64 at a time: on_rows(r0, sl, ty, span) is called by
// every lane once per step with its row r0 + lane: the slot, the tile row and
// the span (empty beyond the last row).
template <int kS, typename Fn>
__device__ __forceinline__ void walk_rows(const RasterParams& P,
                                          WalkSlots<kS>& W, int total,
                                          Fn&& on_rows) {
  const int lane = threadIdx.x & 63;
  const int first = lane < kS ? W.first[lane] : 0x7fffffff;
  for (int r0 = 0; r0 < total; r0 += 64) {
    const int sl = owner_lane(W.own, first, r0);
    const int r = r0 + lane;
    RowSpan span{0, -1, 0x7fffffff, 0x7fffffff};
    int ty = 0;
    if (r < total) {
      ty = W.box[sl].y + (r - W.first[sl]);
      span = row_span(P, W, sl, ty);
    }
    on_rows(r0, sl, ty, span);
  }
}

// One row's hits, as runs of tiles: seg(first tile, tiles).  Lanes run on
// their own rows.
template <int kS, typename Fn>
__device__ __forceinline__ void row_hits(const RasterParams& P,
                                         const WalkSlots<kS>& W, int sl,
                                         int ty, const RowSpan& r, Fn&& seg) {
  if (r.m0 > r.m1) return;
  const int tile0 = W.box[sl].w + ty * P.tiles_x;
  auto live_runs = [&](int t, int n) {
    if (P.live == nullptr) {
      seg((uint32_t)(tile0 + t), (uint32_t)n);
      return;
    }
    for (int i = tile0 + t; i < tile0 + t + n;) {  // word by word
      const int end = min(tile0 + t + n, (i | 31) + 1);
      uint32_t bits = P.live[i >> 5] >> (i & 31);
      if (end - i < 32) bits &= (1u << (end - i)) - 1u;
      while (bits != 0u) {
        const int at = __builtin_ctz(bits);
        const uint32_t rest = ~(bits >> at);
        const int len = rest == 0u ? 32 : __builtin_ctz(rest);
        seg((uint32_t)(i + at), (uint32_t)len);
        bits = at + len >= 32 ? 0u : bits >> (at + len) << (at + len);
      }
      i = end;
    }
  };
  for (int t = r.m0; t <= r.m1; ++t) {
    if (t == r.c0) {
      live_runs(r.c0, r.c1 - r.c0 + 1);
      t = r.c1;
    } else if (tile_hit(P, W, sl, t, ty)) {
      live_runs(t, 1);
    }
  }
}

// Adds seg to the two copies of an LDS histogram of tile digits, cut where
// the digit changes.
__device__ __forceinline__ void add_digits(uint32_t* hist, int shift,
                                           uint32_t t0, uint32_t n) {
  uint32_t* const h = hist + (threadIdx.x & 1) * 257;
  const uint32_t t1 = t0 + n;
  while (t0 < t1) {
    const uint32_t end = min(t1, ((t0 >> shift) + 1u) << shift);
    atomicAdd(&h[(t0 >> shift) & 255u], end - t0);
    t0 = end;
  }
}

// Hands out the wavefront's hits 64 at a time: the rows' spans of a step are
// laid end to end and the lanes take consecutive tiles, so that the wavefront
// writes consecutive pairs.  on_step(hm, hit, sl, tile) is called by every
// lane once per 64 tiles, hm being the ballot of hits (sl and tile mean
// nothing without a hit).  Spans are enumerated splat by splat, so the hits
// before a position are counted with one running total and a lane-masked
// popcount.
template <int kS, typename Fn>
__device__ __forceinline__ void walk_hits(const RasterParams& P,
                                          WalkSlots<kS>& W, int total,
                                          Fn&& on_step) {
  const int lane = threadIdx.x & 63;
  walk_rows(P, W, total, [&](int, int sl, int ty, const RowSpan& r) {
    const int n = max(r.m1 - r.m0 + 1, 0);
    const int inc = wave_prefix_sum(n);
    const int start = inc - n;
    const int tiles = __builtin_amdgcn_readlane(inc, 63);
    const int tile0 = W.box[sl].w + ty * P.tiles_x + r.m0;
    const bool unsure = n > 0 && (r.c0 != r.m0 || r.c1 != r.m1);
    const bool any_unsure = __ballot(unsure) != 0ull;  // uniform
    for (int e0 = 0; e0 < tiles; e0 += 64) {
      const int ow = owner_lane(W.own, start, e0);
      const int off = e0 + lane - __shfl(start, ow, 64);
      const int tile = __shfl(tile0, ow, 64) + off;
      const int osl = __shfl(sl, ow, 64);
      bool hit = e0 + lane < tiles;
      if (any_unsure) {
        const int tx = __shfl(r.m0, ow, 64) + off, oy = __shfl(ty, ow, 64);
        const int c0 = __shfl(r.c0, ow, 64), c1 = __shfl(r.c1, ow, 64);
        if (hit && (tx < c0 || tx > c1)) hit = tile_hit(P, W, osl, tx, oy);
      }
      if (P.live != nullptr && hit)
        hit = ((P.live[tile >> 5] >> (tile & 31)) & 1u) != 0u;
      on_step(__ballot(hit), hit, osl, tile);
    }
  });
}

// Hits among the lanes below `rel` of a step's hit ballot hm (rel in 0..64).
__device__ __forceinline__ int hits_below(uint64_t hm, int rel) {
  return __popcll(rel >= 64 ? hm : (hm & ((1ull << rel) - 1ull)));
}

// LDS of a count block of kW wavefronts of kS splats.
template <int kW, int kS>
struct CountLds {
  WalkSlots<kS> walk[kW];
  int wsum[kW];
};

// The original index that the record of depth rank gid carries.
__device__ __forceinline__ int source_of(const float4* __restrict__ packed,
                                         int gid) {
  return (int)(__float_as_uint(packed[kRecordVec4 * (int64_t)gid + 2].y) &
               0x7fffffffu);
}

// The record of splat orig at depth rank gid.
__device__ __forceinline__ void pack_record(
    const RasterParams& P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ colors,
    const float* __restrict__ opacities, float4* __restrict__ packed, int gid,
    int orig) {
  store_record(packed, gid,
               record_of(P, means2d, conics, colors, opacities, orig,
                         (uint32_t)(P.orig_map != nullptr ? P.orig_map[orig]
                                                          : orig)));
}

// Count block vb of nvb (kW wavefronts, kS splats each), original
// order: splat_count[orig] = tile hits of splat orig and, with block_sums,
// block_sums[vb] = the block's total; with rec_orig also the splat's record
// in original order, its count in the slot (pack_kernel then copies one
// 64-byte record per splat instead of gathering five attribute arrays).
// The blocks also zero zero_words[0..n_zero_words) (grid-stride; read only
// by later launches).  With lds_hist (2 x 257 words of LDS) the block also
// counts its hits' tile digits ((tile >> hist_shift) & 255) and writes them
// to hist_row[0..255]: the pair sort's histogram, in partials that a later
// launch sums (it counts every hit, the emit only those below its capacity:
// the two differ only when the capacity is short, and then the binning is
// redone).
template <int kW, int kS>
__device__ __forceinline__ void count_block(
    const RasterParams& P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ opacities,
    const float* __restrict__ colors, float4* __restrict__ rec_orig,
    int32_t* __restrict__ splat_count, int32_t* __restrict__ block_sums,
    uint32_t* __restrict__ zero_words, int64_t n_zero_words, int vb, int nvb,
    CountLds<kW, kS>& S, uint32_t* lds_hist = nullptr,
    uint32_t* __restrict__ hist_row = nullptr, int hist_shift = 0) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int64_t i = (int64_t)vb * (64 * kW) + threadIdx.x; i < n_zero_words;
       i += (int64_t)nvb * (64 * kW))
    zero_words[i] = 0u;
  if (lds_hist != nullptr) {
    for (int i = threadIdx.x; i < 2 * 257; i += 64 * kW) lds_hist[i] = 0u;
    __syncthreads();
  }
  const int orig = (vb * kW + wave) * kS + lane;
  const bool valid = lane < kS && orig < P.num_splats;
  const int o = valid ? orig : P.num_splats - 1;
  SplatGeom s;
  s.mx = means2d[2 * o + 0];
  s.my = means2d[2 * o + 1];
  s.a = conics[3 * o + 0];
  s.b = conics[3 * o + 1];
  s.c = conics[3 * o + 2];
  s.o = opacities[o];
  WalkSlots<kS>& W = S.walk[wave];
  const int total =
      walk_setup(P, valid, s, o / P.gpb,
                 P.orig_map != nullptr ? P.orig_map[o] : o, W);
  // Hits before the end of this lane's splat's rows (lanes below kS): the
  // running total of the steps before plus the hits of the step's rows below
  // the end; a splat's count is the difference to the previous lane's.
  const int my_end = lane < kS ? W.cend[lane] : 0;
  int run = 0, hits_to_end = 0;
  walk_rows(P, W, total, [&](int r0, int sl, int ty, const RowSpan& r) {
    int n = 0;
    row_hits(P, W, sl, ty, r, [&](uint32_t t0, uint32_t k) {
      n += (int)k;
      if (lds_hist != nullptr) add_digits(lds_hist, hist_shift, t0, k);
    });
    const int inc = wave_prefix_sum(n);
    const int rel = my_end - r0;
    const int below = __shfl(inc, min(max(rel - 1, 0), 63), 64);
    if (rel > 0 && rel <= 64) hits_to_end = run + below;
    run += __builtin_amdgcn_readlane(inc, 63);
  });
  if (lds_hist != nullptr) {
    __syncthreads();
    if (threadIdx.x < 256)
      hist_row[threadIdx.x] = lds_hist[threadIdx.x] + lds_hist[257 + threadIdx.x];
  }
  const int prev_end = __shfl_up(hits_to_end, 1, 64);
  const int n = valid ? hits_to_end - (lane == 0 ? 0 : prev_end) : 0;
  if (valid) splat_count[orig] = n;
  // (the attributes are read again here rather than kept across the walk)
  if (valid && rec_orig != nullptr)
    store_record(rec_orig, orig,
                 record_of(P, means2d, conics, colors, opacities, orig,
                           (uint32_t)n));
  if (block_sums == nullptr) return;
  int v = n;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if (lane == 0) S.wsum[wave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
#pragma unroll
    for (int w = 0; w < kW; ++w) t += S.wsum[w];
    block_sums[vb] = t;
  }
}

__global__ __launch_bounds__(kThreads) void count_kernel(
    RasterParams P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ opacities,
    const float* __restrict__ colors, float4* __restrict__ rec_orig,
    int32_t* __restrict__ splat_count, int32_t* __restrict__ block_sums,
    uint32_t* __restrict__ zero_words, int64_t n_zero_words) {
  __shared__ CountLds<kWaves, kWalkSplats> S;
  count_block<kWaves, kWalkSplats>(P, means2d, conics, opacities, colors, rec_orig,
                      splat_count, block_sums, zero_words, n_zero_words,
                      (int)blockIdx.x, (int)gridDim.x, S);
}

// The count next to the run step of the small-image depth order, in one
// launch: workgroups below run_blocks sort one depth run each (a few CUs for
// most of the launch), the others are count blocks of kRunWaves wavefronts
// and fill the remaining CUs.  The two parts touch disjoint memory.
template <int kS>
union CountRunsLds {
  run_step::RunSortLds runs;
  CountLds<run_step::kRunWaves, kS> count;
};

template <int kS>
__global__ __launch_bounds__(run_step::kRunThreads) void count_depth_runs_kernel(
    RasterParams P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ opacities,
    int32_t* __restrict__ splat_count, uint32_t* __restrict__ zero_words,
    int64_t n_zero_words, const float* __restrict__ depths, int runs,
    int run_blocks, run_step::RunBuffers runs_out, CountHist H) {
  __shared__ CountRunsLds<kS> S;
  __shared__ uint32_t hist[2 * 257];
  if ((int)blockIdx.x < run_blocks) {
    run_step::run_sort_block(depths, P.gpb, runs, (int)blockIdx.x, runs_out,
                             S.runs);
    return;
  }
  const int vb = (int)blockIdx.x - run_blocks;
  count_block<run_step::kRunWaves, kS>(
      P, means2d, conics, opacities, nullptr, nullptr, splat_count, nullptr,
      zero_words, n_zero_words, vb, (int)gridDim.x - run_blocks, S.count,
      H.parts != nullptr ? hist : nullptr,
      H.parts != nullptr ? H.parts + (int64_t)vb * 256 : nullptr, H.shift);
}

// One workgroup: *pair_count = sum of the n block sums (-1 if it does not fit
// in int32).
__global__ __launch_bounds__(kThreads) void sum_kernel(
    const int32_t* __restrict__ block_sums, int n, int32_t* pair_count) {
  __shared__ long long part[kThreads];
  // eight independent loads in flight per thread
  long long acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int i = threadIdx.x;
  for (; i + 7 * kThreads < n; i += 8 * kThreads) {
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] += block_sums[i + u * kThreads];
  }
  for (; i < n; i += kThreads) acc[0] += block_sums[i];
  long long v = 0;
#pragma unroll
  for (int u = 0; u < 8; ++u) v += acc[u];
  part[threadIdx.x] = v;
  __syncthreads();
  for (int half = kThreads / 2; half > 0; half >>= 1) {
    if (threadIdx.x < half) part[threadIdx.x] += part[threadIdx.x + half];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const long long total = part[0];
    *pair_count = total > 0x7fffffffLL ? -1 : (int32_t)total;
  }
}

// Rank step of the small-image depth order with the records packed where
// the ranks land: perm[gid] = in-image index, the record of gid and
// gid_count[gid] = splat_count[orig] (the pair offsets are then scanned by
// emit_kernel<true>).
// Emit workgroups whose totals a rank_pack workgroup adds in LDS first (its
// 256 gids are increasing and usually span a few dozen of them).
constexpr int kAggBlocks = 512;

__global__ __launch_bounds__(run_step::kRankBlock) void rank_pack_kernel(
    RasterParams P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ colors,
    const float* __restrict__ opacities, run_step::RunBuffers runs_in,
    int runs, const int32_t* __restrict__ splat_count,
    int32_t* __restrict__ perm, float4* __restrict__ packed,
    int32_t* __restrict__ gid_count, uint32_t* __restrict__ block_totals,
    int emit_splats, CountHist H) {
  __shared__ run_step::RankLds S;
  __shared__ uint32_t agg[kAggBlocks];
  __shared__ int agg_first;
  const int t = threadIdx.x;
  if (H.parts != nullptr && blockIdx.x == gridDim.x - 1) {
    // the extra workgroup: the pair sort's histogram from the count blocks'
    // partials (kRankSplit thread groups per digit, then their sums in LDS)
    constexpr int kGroups = run_step::kRankBlock / 256;
    uint32_t* red = reinterpret_cast<uint32_t*>(&S);
    const int d = t & 255, g = t >> 8;
    // (eight independent loads in flight per thread)
    uint32_t acc[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    int r = g;
    for (; r + 7 * kGroups < H.nparts; r += 8 * kGroups) {
#pragma unroll
      for (int u = 0; u < 8; ++u) acc[u] += H.parts[(int64_t)(r + u * kGroups) * 256 + d];
    }
    for (; r < H.nparts; r += kGroups) acc[0] += H.parts[(int64_t)r * 256 + d];
    uint32_t v = 0u;
#pragma unroll
    for (int u = 0; u < 8; ++u) v += acc[u];
    red[g * 256 + d] = v;
    __syncthreads();
    if (t < 256) {
      uint32_t sum = 0u;
#pragma unroll
      for (int k = 0; k < kGroups; ++k) sum += red[k * 256 + t];
      H.ghist[t] = sum;
    }
    return;
  }
  if (t < kAggBlocks) agg[t] = 0u;  // (rank_block synchronises before use)
  int my_gid = -1, my_n = 0;
  run_step::rank_block(
      runs_in.keys, runs_in.vals, runs_in.samples, P.gpb, runs,
      (int)blockIdx.x, S, [&](int64_t base, int pos, uint32_t v) {
        const int gid = (int)base + pos;
        const int orig = (int)base + (int)v;
        perm[gid] = (int32_t)v;
        pack_record(P, means2d, conics, colors, opacities, packed, gid, orig);
        my_n = splat_count[orig];
        gid_count[gid] = my_n;
        my_gid = gid;
      });
  // Each gid's count goes to its emit workgroup's total (the emit's later
  // workgroups start from these): the chunk's element 0 has its smallest
  // gid, so workgroups first .. first + kAggBlocks - 1 are summed in LDS,
  // any further one directly.
  if (t == 0) agg_first = my_gid / emit_splats;
  __syncthreads();
  const int first = agg_first;
  if (my_gid >= 0 && my_n != 0) {
    const int wb = my_gid / emit_splats;
    if (wb - first < kAggBlocks)
      atomicAdd(&agg[wb - first], (uint32_t)my_n);
    else
      atomicAdd(&block_totals[wb], (uint32_t)my_n);
  }
  __syncthreads();
  if (t < kAggBlocks && agg[t] != 0u) atomicAdd(&block_totals[first + t], agg[t]);
}

// One thread per depth-sorted splat (gid): gathers the attributes of
// orig = perm[gid] into the packed 64-byte record and turns the per-gid
// tile-hit counts into exclusive offsets splat_offsets in the same launch
// (workgroup scan + decoupled look-back).  splat_offsets[num_splats] = N, or
// -1 when N does not fit in int32 (the offsets are then unusable).  With
// orig_slot also orig_slot[orig] = {offset, gid} (the original-order emit's).
__global__ __launch_bounds__(kThreads) void pack_kernel(
    RasterParams P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ colors,
    const float* __restrict__ opacities, const uint32_t* __restrict__ perm,
    const int32_t* __restrict__ splat_count,
    const float4* __restrict__ rec_orig, float4* __restrict__ packed,
    int32_t* __restrict__ splat_offsets, uint64_t* scan_status,
    uint32_t* scan_ticket, uint32_t* err, int2* __restrict__ orig_slot) {
  __shared__ int wsum[kThreads / 64];
  __shared__ long long s_prefix;
  const int vb = take_ticket(scan_ticket);
  const int gid = vb * kThreads + threadIdx.x;
  int n = 0, orig = 0;
  if (gid < P.num_splats) {
    const int batch = gid / P.gpb;
    // (perm is in [0, G) unless a look-back of the depth sort gave up; the
    // clamp keeps the gathers in bounds then, and the status reports it)
    orig = batch * P.gpb + (int)min(perm[gid], (uint32_t)(P.gpb - 1));
    if (rec_orig != nullptr) {  // the count's record: orig replaces the count
      Record r;
#pragma unroll
      for (int k = 0; k < kRecordVec4; ++k)
        r.v[k] = rec_orig[(int64_t)kRecordVec4 * orig + k];
      const uint32_t slot = __float_as_uint(r.v[2].y);
      n = (int)(slot & 0x7fffffffu);
      const int source = P.orig_map != nullptr ? P.orig_map[orig] : orig;
      r.v[2].y = __uint_as_float((uint32_t)source | (slot & 0x80000000u));
      store_record(packed, gid, r);
    } else {
      pack_record(P, means2d, conics, colors, opacities, packed, gid, orig);
      n = splat_count[orig];
    }
  }
  // Workgroup exclusive scan of the counts.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = n;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(inc, off, 64);
    if (lane >= off) inc += y;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int pre = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) {
    pre += (w < wave) ? wsum[w] : 0;
    total += wsum[w];
  }
  if (wave == 0) {
    if (lane == 0)
      status_store(&scan_status[vb], (vb == 0 ? kFlagInc64 : kFlagAgg64) |
                                         (uint64_t)(uint32_t)total);
    uint64_t prefix = 0;
    if (vb > 0) {
      prefix = lookback64_wave(scan_status, vb, err);
      if (lane == 0)
        status_store(&scan_status[vb], kFlagInc64 | (prefix + (uint32_t)total));
    }
    if (lane == 0) s_prefix = (long long)prefix;
  }
  __syncthreads();
  const long long end = s_prefix + pre + inc;
  if (gid < P.num_splats) {
    splat_offsets[gid] = (int)(end - n);
    if (orig_slot != nullptr) orig_slot[orig] = make_int2((int)(end - n), gid);
  }
  if (gid == P.num_splats - 1)
    splat_offsets[P.num_splats] = end > 0x7fffffffLL ? -1 : (int)end;
}

// The records of splats already in depth order (orig = gid), for callers
// that hold the depth-sorted flat attribute arrays themselves (the
// reference's op roles take those arrays, not packed records).
__global__ __launch_bounds__(kThreads) void pack_records_kernel(
    RasterParams P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ colors,
    const float* __restrict__ opacities, float4* __restrict__ packed) {
  const int gid = (int)blockIdx.x * kThreads + (int)threadIdx.x;
  if (gid < P.num_splats)
    pack_record(P, means2d, conics, colors, opacities, packed, gid, gid);
}

// emit_kernel<false, true>: the walk in original order over the count's
// records.
struct EmitOrig {
  const float4* rec;       // the count's original-order records (hit count
                           // in the slot)
  const int2* slot;        // per orig: {pair offset, gid} (pack_kernel)
};

// emit_kernel<true>: the pair offsets are scanned by the emit itself.
struct EmitScan {
  const int32_t* gid_count;     // per-gid tile-hit counts
  int32_t* splat_offsets;       // written: exclusive offsets; [num_splats] = N
                                // (-1 when N does not fit in int32)
  const uint32_t* block_totals; // per emit workgroup: the sum of its gids'
                                // counts (added by rank_pack_kernel)
};

// One pair: (tile, gid) into keys and vals, or, for the two-pass sort of
// tiles below 2^16 and gids below 2^24 (key_bytes), the word
// (tile >> 8) << 24 | gid into keys and the tile's low byte into key_bytes
// (5 bytes instead of 8).
__device__ __forceinline__ void put_pair(uint32_t* __restrict__ keys,
                                         uint32_t* __restrict__ vals,
                                         uint8_t* __restrict__ key_bytes,
                                         int64_t pos, uint32_t tile,
                                         uint32_t gid) {
  if (key_bytes != nullptr) {
    keys[pos] = ((tile >> 8) << 24) | gid;
    key_bytes[pos] = (uint8_t)tile;
  } else {
    keys[pos] = tile;
    vals[pos] = gid;
  }
}

// Pairs are written (and counted in the histograms) only at positions below
// min(N, capacity): with a capacity below N the output is the first
// `capacity` pairs, consistently.  kScan: each workgroup scans its gids'
// counts, starting from the totals of the workgroups before it (their sum:
// no look-back, no order among workgroups), and writes splat_offsets before
// walking (the offsets, not N, bound the positions then: every pair lies
// below N by construction).  Otherwise splat_offsets (and N in
// splat_offsets[num_splats]) come from pack_kernel.  kOrig (not with kScan):
// the workgroups walk the splats in original order, the count's walk, from
// its records (eo.rec): a splat's pairs start at eo.slot[orig].x.
template <bool kScan, bool kOrig, int kS>
__global__ __launch_bounds__(kThreads) void emit_kernel(
    RasterParams P, const float4* __restrict__ packed,
    const int32_t* __restrict__ splat_offsets, int64_t capacity,
    uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
    uint8_t* __restrict__ key_bytes, int pair_passes, int hist_shift,
    uint32_t* __restrict__ hist_partials,
    uint32_t* ghist_direct, uint32_t* pair_status, int64_t pair_status_words,
    EmitScan sc, EmitOrig eo) {
  static_assert(!(kScan && kOrig), "one source of offsets");
  __shared__ WalkSlots<kS> walk[kWaves];
  __shared__ int base[kWaves][kS];
  // kOrig: per splat its first position less the wavefront's hits before it,
  // and its gid
  __shared__ int wbase[kOrig ? kWaves : 1][kS];
  __shared__ int wgid[kOrig ? kWaves : 1][kS];
  // the pair sort's digit histograms in kHistCopies copies (lane l adds to
  // copy l % kHistCopies; rows 257 words apart, so that one digit's copies
  // lie in different LDS banks): hits of one tile row share the row's
  // digit, and a copy per lane group divides their serialisation
  __shared__ uint32_t h[4][kHistCopies][257];
  __shared__ int wsum[kWaves];
  __shared__ long long wbefore[kWaves];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // (1) zero the pair sort's look-back status (grid-stride)
  for (int64_t i = (int64_t)blockIdx.x * kThreads + t; i < pair_status_words;
       i += (int64_t)gridDim.x * kThreads)
    pair_status[i] = 0u;
  for (int i = t; i < 4 * kHistCopies * 257; i += kThreads) (&h[0][0][0])[i] = 0u;
  const int vb = (int)blockIdx.x;
  __syncthreads();
  // (2) pair emission (gid: the splat's index in the walk's order, its
  // original index with kOrig)
  const int gid = (vb * kWaves + wave) * kS + lane;
  const bool valid = lane < kS && gid < P.num_splats;
  const int g = valid ? gid : P.num_splats - 1;
  const float4* __restrict__ src = kOrig ? eo.rec : packed;
  const float4 p0 = src[kRecordVec4 * (int64_t)g + 0];
  const float4 p1 = src[kRecordVec4 * (int64_t)g + 1];
  const SplatGeom s{p0.x, p0.y, p0.z, p0.w, p1.x, p1.y};
  WalkSlots<kS>& W = walk[wave];
  int64_t n_eff;
  int total;
  if (kScan) {
    // exclusive offsets of the workgroup's gids: wavefront scans, the
    // workgroup's scan, and the totals of the workgroups before it (loaded
    // first, summed after the walk set-up, which overlaps their latency).
    const int n = valid ? sc.gid_count[gid] : 0;
    long long before = 0;
    for (int j = t; j < vb; j += kThreads) before += sc.block_totals[j];
    int inc = n;
#pragma unroll
    for (int off = 1; off < kS; off <<= 1) {
      const int y = __shfl_up(inc, off, 64);
      if (lane >= off) inc += y;
    }
    if (lane == kS - 1) wsum[wave] = inc;
    total = walk_setup(P, valid, s, g / P.gpb,
                       P.live != nullptr ? source_of(src, g) : 0, W);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
    if (lane == 0) wbefore[wave] = before;
    __syncthreads();
    long long pre = 0, wg_before = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      pre += (w < wave) ? wsum[w] : 0;
      wg_before += wbefore[w];
    }
    const long long end = wg_before + pre + inc;
    if (valid) {
      sc.splat_offsets[gid] = (int)(end - n);
      // positions at or above the capacity are not written: clamp there
      base[wave][lane] = (int)min((long long)capacity, end - n);
    }
    // (lanes 32..63 alias the next wavefront's gids: only a valid lane
    // writes)
    if (valid && gid == P.num_splats - 1)
      sc.splat_offsets[P.num_splats] = end > 0x7fffffffLL ? -1 : (int)end;
    n_eff = capacity;
  } else if (kOrig) {
    const int n =
        valid ? (int)(__float_as_uint(src[kRecordVec4 * (int64_t)g + 2].y) &
                      0x7fffffffu)
              : 0;
    const int2 sg = valid ? eo.slot[g] : make_int2(0, 0);
    n_eff = min(capacity, (int64_t)max(splat_offsets[P.num_splats], 0));
    total = walk_setup(P, valid, s, g / P.gpb,
                       P.orig_map != nullptr ? P.orig_map[g] : g, W);
    // hits of the wavefront's splats up to this one
    int inc = n;
#pragma unroll
    for (int off = 1; off < kS; off <<= 1) {
      const int y = __shfl_up(inc, off, 64);
      if (lane >= off) inc += y;
    }
    if (lane < kS) {
      wbase[kOrig ? wave : 0][lane] = sg.x - (inc - n);
      wgid[kOrig ? wave : 0][lane] = sg.y;
    }
  } else {
    if (lane < kS) base[wave][lane] = splat_offsets[g];
    n_eff = min(capacity, (int64_t)max(splat_offsets[P.num_splats], 0));
    total = walk_setup(P, valid, s, g / P.gpb,
                       P.live != nullptr ? source_of(src, g) : 0, W);
  }
  const int gid0 = gid - lane;
  // The wavefront's splats own consecutive ranges starting at the first
  // one's offset, and the hits arrive in splat order: a hit's position is
  // that offset plus the hits before it.
  const int64_t wave_base = kOrig ? 0 : base[wave][0];
  int64_t run = 0;
  walk_hits(P, W, total, [&](uint64_t hm, bool hit, int sl, int tile) {
    const int64_t pos =
        (kOrig ? (hit ? (int64_t)wbase[kOrig ? wave : 0][sl] : 0) : wave_base) +
        run + hits_below(hm, lane);
    run += __popcll(hm);
    // (pos >= 0 whenever n_eff > 0, unless a look-back of the depth sort
    // gave up and left the original-order offsets unwritten)
    if (hit && pos < n_eff && (!kOrig || pos >= 0)) {
      put_pair(keys, vals, key_bytes, pos, (uint32_t)tile,
               kOrig ? (uint32_t)wgid[kOrig ? wave : 0][sl]
                     : (uint32_t)(gid0 + sl));
      for (int p = 0; p < pair_passes; ++p)
        atomicAdd(&h[p][lane % kHistCopies]
                     [((uint32_t)tile >> (hist_shift + 8 * p)) & 255u],
                  1u);
    }
  });
  // (3) this workgroup's digit histograms for the pair sort: added to the
  // zeroed global histograms (ghist_direct, few workgroups) or stored as
  // hist_partials[(p * 256 + d) * nblk + workgroup] for hist_reduce_kernel
  __syncthreads();
  for (int p = 0; p < pair_passes; ++p) {
    uint32_t c = 0u;
#pragma unroll
    for (int q = 0; q < kHistCopies; ++q) c += h[p][q][t];
    if (ghist_direct != nullptr) {
      if (c) atomicAdd(&ghist_direct[p * 256 + t], c);
    } else {
      hist_partials[((int64_t)p * 256 + t) * gridDim.x + blockIdx.x] = c;
    }
  }
}

// ghist[p][d] = sum over the emit workgroups of their digit-d counts of pass
// p: one workgroup per (p, d) reads that row of partials contiguously.
__global__ __launch_bounds__(kThreads) void hist_reduce_kernel(
    const uint32_t* __restrict__ hist_partials, int nblk,
    uint32_t* __restrict__ ghist) {
  __shared__ uint32_t part[kThreads / 64];
  const uint32_t* row = hist_partials + (int64_t)blockIdx.x * nblk;
  // eight independent loads in flight per thread
  uint32_t acc[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
  int b = threadIdx.x;
  for (; b + 7 * kThreads < nblk; b += 8 * kThreads) {
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] += row[b + u * kThreads];
  }
  for (; b < nblk; b += kThreads) acc[0] += row[b];
  uint32_t v = 0u;
#pragma unroll
  for (int u = 0; u < 8; ++u) v += acc[u];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0u;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) t += part[w];
    ghist[blockIdx.x] = t;   // blockIdx.x = p * 256 + d
  }
}

// tile_offsets from the sorted tile keys: index i (0 <= i <= n) is the first
// pair of every tile t with keys[i-1] < t <= keys[i] (keys[-1] = -1,
// keys[n] = num_tiles), so tile_offsets[num_tiles] = n.  With n_dev the key
// count is min(*n_dev, n).  Grid-stride over the indices, kRangeUnroll of
// them per iteration with all their loads issued first (indices clamped into
// [0, n_cap), so the loads need no branch), which keeps a launch over 1e8
// keys to a few thousand workgroups.
constexpr int kRangeUnroll = 4;
constexpr int kRangeMaxBlocks = 2048;
struct StatusWords {
  const uint32_t* err[3];  // give-up status words (null: not used)
  int32_t* out;            // their OR (null: not reported)
  int32_t* long_flag;      // null, or a device word (zero before the
                           // launch) set to 1 if a tile range is longer
                           // than kHandoffPairs
  ZeroSpan zero[2];        // zeroed by the launch on the side
};

__global__ __launch_bounds__(kThreads) void ranges_kernel(
    const uint32_t* __restrict__ sorted_keys, int64_t n_cap,
    const int32_t* __restrict__ n_dev, int num_tiles,
    int32_t* __restrict__ tile_offsets, StatusWords sw) {
  // Every look-back of the binning ran in an earlier launch.  If one gave
  // up, the pairs may hold unwritten entries: every tile is emptied instead
  // (the compositors then read no pair), and the status says why.
  uint32_t e = 0u;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (sw.err[k] != nullptr) e |= *sw.err[k];
  if (blockIdx.x == 0 && threadIdx.x == 0 && sw.out != nullptr)
    *sw.out = (int32_t)e;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
#pragma unroll
  for (int z = 0; z < 2; ++z)
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
         i < sw.zero[z].n; i += stride)
      sw.zero[z].p[i] = 0u;
  if (e != 0u) {
    for (int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
         t <= num_tiles; t += stride)
      tile_offsets[t] = 0;
    return;
  }
  const int64_t n = n_dev ? min(n_cap, (int64_t)max(*n_dev, 0)) : n_cap;
  bool long_range = false;  // a range starting here exceeds kHandoffPairs
  for (int64_t i0 = (int64_t)blockIdx.x * kThreads + threadIdx.x; i0 <= n;
       i0 += kRangeUnroll * stride) {
    uint32_t kp[kRangeUnroll], kc[kRangeUnroll];
#pragma unroll
    for (int u = 0; u < kRangeUnroll; ++u) {
      const int64_t i = min(i0 + u * stride, n);
      kp[u] = sorted_keys[max(i - 1, (int64_t)0)];
      kc[u] = sorted_keys[max(min(i, n - 1), (int64_t)0)];
    }
#pragma unroll
    for (int u = 0; u < kRangeUnroll; ++u) {
      const int64_t i = i0 + u * stride;
      if (i > n) break;
      const int64_t prev = (i == 0) ? -1 : (int64_t)kp[u];
      const int64_t cur = (i == n) ? (int64_t)num_tiles
                                   : min((int64_t)kc[u], (int64_t)num_tiles);
      for (int64_t t = prev + 1; t <= cur; ++t) tile_offsets[t] = (int32_t)i;
      // tile cur's range starts at i: longer than kHandoffPairs iff its
      // key is still there kHandoffPairs places on
      if (sw.long_flag != nullptr && prev != cur && i + kHandoffPairs < n)
        long_range |= sorted_keys[i + kHandoffPairs] == kc[u];
    }
  }
  if (sw.long_flag != nullptr && __ballot(long_range) != 0ull &&
      (threadIdx.x & 63) == 0)
    *sw.long_flag = 1;
}

// After radix_pair_sort_ranges wrote every tile_offsets entry: the
// binning's status, empty ranges (all zero) when a look-back gave up or no
// pair was emitted, the long-range flag and the zero spans, as ranges_kernel
// does beside its ranges.
__global__ __launch_bounds__(kThreads) void ranges_finish_kernel(
    int64_t n_cap, const int32_t* __restrict__ n_dev, int num_tiles,
    int32_t* __restrict__ tile_offsets, StatusWords sw) {
  uint32_t e = 0u;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (sw.err[k] != nullptr) e |= *sw.err[k];
  if (blockIdx.x == 0 && threadIdx.x == 0 && sw.out != nullptr)
    *sw.out = (int32_t)e;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  const int64_t first = (int64_t)blockIdx.x * kThreads + threadIdx.x;
#pragma unroll
  for (int z = 0; z < 2; ++z)
    for (int64_t i = first; i < sw.zero[z].n; i += stride) sw.zero[z].p[i] = 0u;
  const int64_t n = n_dev ? min(n_cap, (int64_t)max(*n_dev, 0)) : n_cap;
  if (e != 0u || n == 0) {
    for (int64_t t = first; t <= num_tiles; t += stride) tile_offsets[t] = 0;
    return;
  }
  bool long_range = false;
  for (int64_t t = first; t < num_tiles; t += stride)
    long_range |= tile_offsets[t + 1] - tile_offsets[t] > kHandoffPairs;
  if (sw.long_flag != nullptr && __ballot(long_range) != 0ull &&
      (threadIdx.x & 63) == 0)
    *sw.long_flag = 1;
}

__global__ void host_report_kernel(HostReport R) {
  if (threadIdx.x == 0) write_host_report(R);
}

// Bucket counting sort (launch_bucket_sort): one workgroup per bucket of
// 2^low_bits tiles, whose pairs the onesweep pass on the higher tile bits
// left contiguous and in gid order.  A pass takes up to kBucketChunk of the
// bucket's pairs: wavefront w the pairs [w*64*R, (w+1)*64*R) of the pass,
// round r of it the 64 from w*64*R + r*64 (R = kBucketRounds), so that the
// order (pass, wavefront, round, lane) is the pairs' order in the bucket.
// A pair's output index is its digit's start, plus the pairs of that digit
// in earlier passes, in earlier wavefronts of its pass, in the lane's earlier
// rounds and in lower lanes of its round (ballot match): a stable sort.  The
// digit starts are the scan of the digit counts: counted by the single pass
// of a bucket of at most kBucketChunk pairs, else by a counting sweep first.
constexpr int kBucketWaves = 16;
constexpr int kBucketThreads = kBucketWaves * 64;
constexpr int kBucketRounds = kBucketChunk / kBucketThreads;

struct BucketLds {
  uint32_t cnt[kBucketWaves][256];  // per-wavefront digit counts, then the
                                    // digit's output index for the wavefront
  uint32_t run[256];                // digit's next output index (sweeps)
  uint32_t wsum[kBucketWaves];
};

// Exclusive scan of v over threads 0..255 of the workgroup (0 elsewhere);
// every thread calls it (it synchronises the workgroup).
__device__ __forceinline__ uint32_t bucket_digit_scan(uint32_t v,
                                                      BucketLds& S) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  uint32_t inc = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(inc, off, 64);
    if (lane >= off) inc += y;
  }
  if (lane == 63 && wave < 4) S.wsum[wave] = inc;
  __syncthreads();
  uint32_t pre = 0u;
#pragma unroll
  for (int w = 0; w < 4; ++w) pre += (w < wave) ? S.wsum[w] : 0u;
  __syncthreads();  // wsum is read before it is written again
  return pre + inc - v;
}

__global__ __launch_bounds__(kBucketThreads) void bucket_sort_kernel(
    BucketSortArgs A) {
  __shared__ BucketLds S;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int b = blockIdx.x;
  const int ndig = 1 << A.low_bits;
  const uint32_t dmask = (uint32_t)ndig - 1u;
  const int tile0 = b << A.low_bits;
  uint32_t e = 0u;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (A.err[k] != nullptr) e |= *A.err[k];
  if (b == 0 && t == 0 && A.status_out != nullptr) *A.status_out = (int32_t)e;
  const int64_t n =
      A.n_dev ? min(A.n, (int64_t)max(*A.n_dev, 0)) : A.n;
  // the bucket's first index, the sizes of buckets 0..b-1 (b < 256), summed
  // by every wavefront (no workgroup barrier)
  uint32_t before = 0u, all = 0u;
#pragma unroll
  for (int i = lane; i < 256; i += 64) {
    const uint32_t v = A.bucket_sizes[i];
    before += (i < b) ? v : 0u;
    all += v;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    before += __shfl_xor(before, off, 64);
    all += __shfl_xor(all, off, 64);
  }
  const uint32_t base = before;
  // (the sizes add up to n by construction; the clamp keeps every access
  // inside the first n pairs regardless)
  const uint32_t size = (uint32_t)min(
      (int64_t)A.bucket_sizes[b], max((int64_t)0, n - (int64_t)base));
  for (int i = t; i < kBucketWaves * 256; i += kBucketThreads)
    (&S.cnt[0][0])[i] = 0u;
  const int64_t stride = (int64_t)gridDim.x * kBucketThreads;
#pragma unroll
  for (int z = 0; z < 2; ++z)
    for (int64_t i = (int64_t)b * kBucketThreads + t; i < A.zero[z].n;
         i += stride)
      A.zero[z].p[i] = 0u;
  // A look-back of the binning gave up: every tile range is empty (as in
  // ranges_kernel).
  if (e != 0u) {
    for (int d = t; d < ndig; d += kBucketThreads) {
      if (tile0 + d >= A.num_tiles) break;
      A.tile_offsets[tile0 + d] = 0;
      if (A.tile_counts != nullptr) A.tile_counts[tile0 + d] = 0;
    }
    if (b == 0 && t == 0) A.tile_offsets[A.num_tiles] = 0;
    return;
  }
  // the end of the last range: the pairs the buckets hold (n by
  // construction), so that no range reaches past the sorted pairs
  if (b == 0 && t == 0)
    A.tile_offsets[A.num_tiles] = (int32_t)min(n, (int64_t)all);
  // An empty bucket (no pairs, or none left below n): its tiles' ranges are
  // empty and start at the bucket's first index (at most n, so that the
  // offsets stay monotone when the buffers hold fewer pairs than the
  // buckets).  The chunk loop below writes the ranges of the other buckets;
  // it does not run for size 0.  (size is the same for the whole workgroup,
  // so no thread waits at a barrier that the others skip.)
  if (size == 0u) {
    const int32_t start = (int32_t)min((int64_t)base, n);
    for (int d = t; d < ndig; d += kBucketThreads) {
      if (tile0 + d >= A.num_tiles) break;
      A.tile_offsets[tile0 + d] = start;
      if (A.tile_counts != nullptr) A.tile_counts[tile0 + d] = 0;
    }
    return;
  }
  const bool sweep = size > (uint32_t)kBucketChunk;
  bool long_range = false;
  if (sweep) {
    // counting sweep, then the digit starts
    if (t < 256) S.run[t] = 0u;
    __syncthreads();
    for (uint32_t i = t; i < size; i += kBucketThreads)
      atomicAdd(&S.run[A.keys[base + i] & dmask], 1u);
    __syncthreads();
    const uint32_t tot = t < 256 ? S.run[t] : 0u;
    const uint32_t first = base + bucket_digit_scan(tot, S);
    if (t < ndig && tile0 + t < A.num_tiles) {
      A.tile_offsets[tile0 + t] = (int32_t)first;
      if (A.tile_counts != nullptr) A.tile_counts[tile0 + t] = (int32_t)tot;
      long_range = tot > (uint32_t)kHandoffPairs;
    }
    if (t < 256) S.run[t] = first;
    __syncthreads();
  }
  const uint64_t lt = run_step::lanes_below();
  for (uint32_t c0 = 0; c0 < size; c0 += kBucketChunk) {
    uint32_t d[kBucketRounds], v[kBucketRounds], rank[kBucketRounds];
    bool ok[kBucketRounds];
#pragma unroll
    for (int r = 0; r < kBucketRounds; ++r) {
      const uint32_t li =
          c0 + (uint32_t)(wave * 64 * kBucketRounds + r * 64 + lane);
      ok[r] = li < size;
      d[r] = ok[r] ? (A.keys[base + li] & dmask) : 0u;
      v[r] = ok[r] ? A.vals[base + li] : 0u;
    }
    __syncthreads();  // the counts are zero
#pragma unroll
    for (int r = 0; r < kBucketRounds; ++r) {
      const uint64_t peers =
          run_step::same_digit_lanes(d[r]) & __builtin_amdgcn_ballot_w64(ok[r]);
      const uint32_t below = (uint32_t)__popcll(peers & lt);
      // every lane of the digit reads the count, then its lowest lane adds
      // the group's size (one wavefront's LDS accesses take effect in
      // program order)
      const uint32_t old = S.cnt[wave][d[r]];
      __builtin_amdgcn_wave_barrier();
      if (ok[r] && below == 0u)
        S.cnt[wave][d[r]] = old + (uint32_t)__popcll(peers);
      rank[r] = old + below;
    }
    __syncthreads();
    // digit t: its wavefronts' output indices
    uint32_t tot = 0u;
    if (t < 256) {
#pragma unroll
      for (int w = 0; w < kBucketWaves; ++w) tot += S.cnt[w][t];
    }
    uint32_t first;
    if (sweep) {
      first = t < 256 ? S.run[t] : 0u;
    } else {
      first = base + bucket_digit_scan(tot, S);
      if (t < ndig && tile0 + t < A.num_tiles) {
        A.tile_offsets[tile0 + t] = (int32_t)first;
        if (A.tile_counts != nullptr) A.tile_counts[tile0 + t] = (int32_t)tot;
        long_range = tot > (uint32_t)kHandoffPairs;
      }
    }
    if (t < 256) {
      uint32_t o = first;
#pragma unroll
      for (int w = 0; w < kBucketWaves; ++w) {
        const uint32_t c = S.cnt[w][t];
        S.cnt[w][t] = o;
        o += c;
      }
      if (sweep) S.run[t] = o;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kBucketRounds; ++r)
      if (ok[r]) A.binned_ids[S.cnt[wave][d[r]] + rank[r]] = v[r];
    if (c0 + kBucketChunk < size) {
      __syncthreads();  // the indices are read before they are cleared
      for (int i = t; i < kBucketWaves * 256; i += kBucketThreads)
        (&S.cnt[0][0])[i] = 0u;
    }
  }
  if (A.long_flag != nullptr && __ballot(long_range) != 0ull && lane == 0)
    *A.long_flag = 1;
}

// ---- The tile-sorted binning (launch_tile_sorted): three launches instead of
// five for scenes of up to 256K splats.  Latency bounds them: a chain of
// dependent loads and LDS steps each, 3 to 9 MB moved.  The splats keep their
// original order, so there is no depth order to wait for (run sort and ranks,
// 30 us of serial chains at 64K splats); instead each pair carries its splat's depth
// key, and the workgroup that groups a bucket's pairs by tile also sorts each
// tile's list by (depth, index), which is the stable depth order.  The pairs
// go straight to their bucket: the count's per-block digit counts, which the
// one-call binning reduces to one histogram, give each emit block its place
// in every bucket, so there is no pass over the pairs and no look-back either.
//
// tile_count_kernel  records in original order, each block's pairs per bucket
// tile_emit_kernel   every block sums the counts of the blocks before it (256
//   buckets x at most 256 blocks), walks again and writes {depth key, tile in
//   the bucket << 24 | index} at its places, in any order inside them
// tile_sort_kernel   a workgroup per bucket: tile counts, grouping and ranks
//   in LDS, the ids and the tile ranges
//
// Measured against the one-call binning (us for count, emit and sort; the five
// launches): 64K splats at 1080p 11.9 + 13.1 + 6.5 against 60 in all, at 4096 x
// 4096 11.8 + 15.9 + 9.3 against 63; 128K splats at 1080p 15.0 + 15.2 + 11.8
// against 83; 5000 splats at 1080p 8.1 + 8.4 + 4.2 against 43; 16K splats at
// 512 x 512 8.7 + 8.7 + 6.1 against 45; two images of 32K splats at 600 x 800
// 10.0 + 12.4 + 8.7 against 55; 262K splats in seven images of 769 x 729 14.8 +
// 19.2 + 26.7 against 122, in four of 1811 x 1632 14.7 + 17.8 + 11.0 against 112.
constexpr int kTileWaves = 16;
constexpr int kTileThreads = 64 * kTileWaves;
// A bucket that the sort's LDS does not hold (128 KB of pairs, 16 in registers
// per thread), a tile list above kTileList, or a bucket whose lists take
// longer to rank (their lengths squared, about 40 us per million, bound by
// the 64-bit compares; two 32-bit subtractions, or four entries per thread
// that share their reads, were slower) than the depth order and the pair sort
// of the one-call binning, sets kTileSkewed in the long-range flag and leaves
// its tiles empty; the caller bins such a scene by the other path.  1.2M
// squares (131K splats at 2000 x 2000, 121 pairs a tile): sort 43 us, 76 in
// all against 120; 1.9M (131K at 1080p, 241 a tile): 72, 106 against 119;
// 60K splats at 745 x 837 (220 a tile, 0.5M): 33, 58 against 76.
constexpr int kTileRounds = kTileBucket / kTileThreads;
constexpr uint32_t kTileWorkSmall = 1u << 20;  // up to 64K splats
constexpr uint32_t kTileWork = 3u << 19;

// The wavefront's splats staged for the walk, in original order.
template <int kS>
__device__ __forceinline__ int tile_walk_setup(
    const RasterParams& P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ opacities,
    int orig, bool valid, WalkSlots<kS>& W) {
  const int o = valid ? orig : P.num_splats - 1;
  SplatGeom s;
  s.mx = means2d[2 * o + 0];
  s.my = means2d[2 * o + 1];
  s.a = conics[3 * o + 0];
  s.b = conics[3 * o + 1];
  s.c = conics[3 * o + 2];
  s.o = opacities[o];
  return walk_setup(P, valid, s, o / P.gpb, o, W);
}

template <int kS>
__global__ __launch_bounds__(kTileThreads) void tile_count_kernel(
    RasterParams P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ colors,
    const float* __restrict__ opacities, float4* __restrict__ packed,
    uint32_t* __restrict__ parts, int shift, int32_t* __restrict__ ctl,
    ZeroSpan z0, ZeroSpan z1) {
  __shared__ WalkSlots<kS> walk[kTileWaves];
  __shared__ uint32_t hist[2 * 257];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t stride = (int64_t)gridDim.x * kTileThreads;
  const int64_t first = (int64_t)blockIdx.x * kTileThreads + t;
  for (int64_t i = first; i < z0.n; i += stride) z0.p[i] = 0u;
  for (int64_t i = first; i < z1.n; i += stride) z1.p[i] = 0u;
  if (first < 4) ctl[first] = 0;
  for (int i = t; i < 2 * 257; i += kTileThreads) hist[i] = 0u;
  __syncthreads();
  const int orig = ((int)blockIdx.x * kTileWaves + wave) * kS + lane;
  const bool valid = lane < kS && orig < P.num_splats;
  WalkSlots<kS>& W = walk[wave];
  const int total =
      tile_walk_setup(P, means2d, conics, opacities, orig, valid, W);
  walk_rows(P, W, total, [&](int, int sl, int ty, const RowSpan& r) {
    row_hits(P, W, sl, ty, r, [&](uint32_t t0, uint32_t n) {
      add_digits(hist, shift, t0, n);
    });
  });
  if (valid)
    store_record(packed, orig,
                 record_of(P, means2d, conics, colors, opacities, orig,
                           (uint32_t)orig));
  __syncthreads();
  if (t < 256) parts[(int64_t)blockIdx.x * 256 + t] = hist[t] + hist[257 + t];
}

template <int kS>
__global__ __launch_bounds__(kTileThreads) void tile_emit_kernel(
    RasterParams P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ opacities,
    const float* __restrict__ depths, const uint32_t* __restrict__ parts,
    int shift, int64_t capacity, uint2* __restrict__ pairs,
    uint32_t* __restrict__ bucket_start, int32_t* __restrict__ ctl) {
  __shared__ WalkSlots<kS> walk[kTileWaves];
  __shared__ uint32_t dkey[kTileWaves][kS];
  __shared__ uint32_t cursor[256];
  __shared__ uint32_t red[2][kTileThreads];
  __shared__ unsigned long long wsum[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int vb = (int)blockIdx.x, nblk = (int)gridDim.x;
  const int orig0 = (vb * kTileWaves + wave) * kS;
  const int orig = orig0 + lane;
  const bool valid = lane < kS && orig < P.num_splats;
  {  // bucket t % 256 in a quarter of the blocks: all, and those before this
    const int d = t & 255, g = t >> 8;
    uint32_t all = 0u, before = 0u;
    for (int r = g; r < nblk; r += 64) {  // sixteen loads in flight
      uint32_t v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u)
        v[u] = parts[(int64_t)min(r + 4 * u, nblk - 1) * 256 + d];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const uint32_t x = r + 4 * u < nblk ? v[u] : 0u;
        all += x;
        before += r + 4 * u < vb ? x : 0u;
      }
    }
    red[0][t] = all;
    red[1][t] = before;
  }
  WalkSlots<kS>& W = walk[wave];
  const int total =
      tile_walk_setup(P, means2d, conics, opacities, orig, valid, W);
  if (lane < kS) dkey[wave][lane] = valid ? depth_key(depths[orig]) : 0u;
  __syncthreads();
  unsigned long long inc = 0;
  uint32_t all = 0u, before = 0u;
  if (t < 256) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      all += red[0][g * 256 + t];
      before += red[1][g * 256 + t];
    }
    inc = all;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned long long y = __shfl_up(inc, off, 64);
    if (lane >= off) inc += y;
  }
  if (t < 256 && lane == 63) wsum[wave] = inc;
  __syncthreads();
  if (t < 256) {
    for (int w = 0; w < wave; ++w) inc += wsum[w];
    // (positions at or above the capacity, below 2^31, are not written)
    const unsigned long long start = inc - all;
    const unsigned long long top = 0x7fffffffull;
    cursor[t] = (uint32_t)min(start + before, top);
    if (vb == 0) {
      bucket_start[t] = (uint32_t)min(start, top);
      if (t == 255) {
        bucket_start[256] = (uint32_t)min(inc, top);
        ctl[0] = inc > top ? -1 : (int32_t)inc;
      }
    }
  }
  __syncthreads();
  const uint32_t low = (1u << shift) - 1u;
  walk_hits(P, W, total, [&](uint64_t, bool hit, int sl, int tile) {
    if (!hit) return;
    const uint32_t pos = atomicAdd(&cursor[((uint32_t)tile >> shift) & 255u], 1u);
    if (pos < (uint32_t)capacity)
      pairs[pos] = make_uint2(dkey[wave][sl], ((uint32_t)tile & low) << 24 |
                                                  (uint32_t)(orig0 + sl));
  });
}

__global__ __launch_bounds__(kTileThreads) void tile_sort_kernel(
    const uint2* __restrict__ pairs, const uint32_t* __restrict__ bucket_start,
    int64_t capacity, int num_tiles, int low_bits, uint32_t most_work,
    uint32_t* __restrict__ binned_ids, int32_t* __restrict__ tile_offsets,
    int32_t* __restrict__ tile_ends, int32_t* __restrict__ ctl) {
  __shared__ uint64_t list[kTileBucket];  // depth key << 32 | tile << 24 | index
  __shared__ uint32_t cnt[256], start[256];
  __shared__ uint32_t wsum[4];
  __shared__ int skewed;
  __shared__ uint32_t work;  // below 2^28: a bucket's lists' lengths squared
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int b = (int)blockIdx.x;
  const int tile0 = b << low_bits, ndig = 1 << low_bits;
  const uint32_t cap = (uint32_t)capacity;
  const uint32_t base = min(bucket_start[b], cap);
  const uint32_t end = min(bucket_start[b + 1], cap);
  const uint32_t size = end - base;
  if (t < 256) cnt[t] = 0u;
  if (t == 0) {
    skewed = size > (uint32_t)kTileBucket;
    work = 0u;
  }
  if (b == (int)gridDim.x - 1 && t == 0) tile_offsets[num_tiles] = (int32_t)end;
  __syncthreads();
  const bool fits = size <= (uint32_t)kTileBucket;
  uint2 v[kTileRounds];
  uint32_t slot[kTileRounds];
  if (fits) {
#pragma unroll
    for (int r = 0; r < kTileRounds; ++r) {
      const uint32_t i = (uint32_t)(t + kTileThreads * r);
      if (i < size) v[r] = pairs[base + i];
    }
#pragma unroll
    for (int r = 0; r < kTileRounds; ++r) {
      const uint32_t i = (uint32_t)(t + kTileThreads * r);
      if (i < size) slot[r] = atomicAdd(&cnt[v[r].y >> 24], 1u);
    }
  }
  __syncthreads();
  const uint32_t n = t < 256 ? cnt[t] : 0u;
  uint32_t inc = n;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(inc, off, 64);
    if (lane >= off) inc += y;
  }
  if (t < 256) {
    if (lane == 63) wsum[wave] = inc;
    if (n > (uint32_t)kTileList) skewed = 1;
    if (n > 0u) atomicAdd(&work, n * n);
  }
  __syncthreads();
  const bool skip = skewed != 0 || work > most_work;  // uniform
  if (t < 256) {
    for (int w = 0; w < wave; ++w) inc += wsum[w];
    start[t] = inc - n;
    // (a skewed bucket's tiles are empty, at its end; the tile before them
    // ends at the bucket's base, which only its tile_ends says)
    if (t < ndig && tile0 + t < num_tiles) {
      tile_offsets[tile0 + t] = (int32_t)(skip ? end : base + inc - n);
      tile_ends[tile0 + t] = (int32_t)(skip ? end : base + inc);
    }
    const bool is_long = n > (uint32_t)kHandoffPairs;
    if (__ballot(is_long) != 0ull && lane == 0) atomicOr(ctl + 2, 1);
  }
  if (skip) {
    if (t == 0) atomicOr(ctl + 2, kTileSkewed);
    return;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kTileRounds; ++r) {
    const uint32_t i = (uint32_t)(t + kTileThreads * r);
    if (i < size)
      list[start[v[r].y >> 24] + slot[r]] = (uint64_t)v[r].x << 32 | v[r].y;
  }
  __syncthreads();
  // Each entry's rank in its tile (the entries' tiles agree, so the low words
  // compare by index); neighbouring threads mostly share a tile, and read
  // the same words.
  for (uint32_t i = t; i < size; i += kTileThreads) {
    const uint64_t own = list[i];
    const uint32_t d = (uint32_t)own >> 24;
    const uint32_t s0 = start[d], s1 = s0 + cnt[d];
    uint32_t rank = 0u, j = s0;
    for (; j + 4 <= s1; j += 4) {
      rank += (uint32_t)(list[j] < own);
      rank += (uint32_t)(list[j + 1] < own);
      rank += (uint32_t)(list[j + 2] < own);
      rank += (uint32_t)(list[j + 3] < own);
    }
    for (; j < s1; ++j) rank += (uint32_t)(list[j] < own);
    binned_ids[base + s0 + rank] = (uint32_t)own & 0xffffffu;
  }
}

__global__ __launch_bounds__(kThreads) void counts_kernel(
    const int32_t* __restrict__ tile_offsets, int num_tiles,
    int32_t* __restrict__ tile_counts) {
  const int t = blockIdx.x * kThreads + threadIdx.x;
  if (t < num_tiles) tile_counts[t] = tile_offsets[t + 1] - tile_offsets[t];
}

__global__ void fill_i32_kernel(int32_t* dst, int32_t v, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = v;
}

__global__ void fill_f32_kernel(float* dst, float v, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = v;
}

// Zeroes two word ranges in one launch (grid-stride).
__global__ void zero2_kernel(uint32_t* a, int64_t na, uint32_t* b, int64_t nb) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
       i < na || i < nb; i += stride) {
    if (i < na) a[i] = 0u;
    if (i < nb) b[i] = 0u;
  }
}

// Zeroes the four per-splat gradient arrays (2n, 3n, 3n, n floats) in one
// launch.
__global__ void zero_grads_kernel(float* g_m, float* g_q, float* g_c,
                                  float* g_o, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 2 * n) g_m[i] = 0.0f;
  if (i < 3 * n) {
    g_q[i] = 0.0f;
    g_c[i] = 0.0f;
  }
  if (i < n) g_o[i] = 0.0f;
}

}  // namespace

int count_blocks(const RasterParams& P) {
  return (P.num_splats + kWalkBlockSplats - 1) / kWalkBlockSplats;
}

int launch_count(const RasterParams& P, const float* means2d,
                 const float* conics, const float* opacities,
                 int32_t* splat_count, int32_t* block_sums,
                 int32_t* pair_count, uint32_t* zero_words,
                 int64_t n_zero_words, hipStream_t stream,
                 const float* colors, float* rec_orig) {
  const int nblk = count_blocks(P);
  launch_traced("count_kernel", count_kernel, dim3((unsigned)nblk),
                dim3(kThreads), 0, stream, P, means2d, conics, opacities,
                colors, reinterpret_cast<float4*>(rec_orig), splat_count,
                block_sums, zero_words, n_zero_words);
  int rc = check_launch("count_kernel");
  if (rc || pair_count == nullptr) return rc;
  launch_traced("sum_kernel", sum_kernel, dim3(1), dim3(kThreads), 0, stream,
                block_sums, nblk, pair_count);
  return check_launch("sum_kernel");
}

// Splats of many tiles each: a wavefront of 32 of them walks for long while
// few wavefronts run (two images of 100K 3D splats at 29 pairs per splat:
// emit 80 us with 32, 68 with 16 when every tile was tested, 45 with 16 now),
// and with few splats in all fewer per wavefront only fill the chip (512
// splats: emit 8.5 us with 32, 6.6 with 16).  64K splats of 5 to 13 pairs are as fast or faster with 32 (their
// rank launch adds to more totals otherwise, 15 against 22 us).  No fewer than
// keep the emit launch within kScanEmitMaxBlocks workgroups: with more the
// batch would leave the small-image path (binning of four images of 131,000
// splats at 25 pairs each 338 us, 406 outside it; of three of 100,003 243, 285).
constexpr int kFewSplatPairs = 24;
constexpr int kFewSplats = 1 << 14;

int walk_splats(const RasterParams& P, int64_t capacity) {
  if (capacity >= (int64_t)kFewSplatPairs * P.num_splats)
    for (int walk = 8; walk <= 16; walk *= 2)
      if (emit_blocks(P, walk) <= kScanEmitMaxBlocks) return walk;
  return P.num_splats <= kFewSplats ? 16 : kWalkSplats;
}

int count_depth_runs_blocks(const RasterParams& P, int walk) {
  const int per_block = run_step::kRunWaves * walk;
  return (P.num_splats + per_block - 1) / per_block;
}

int launch_count_depth_runs(const RasterParams& P, const float* means2d,
                            const float* conics, const float* opacities,
                            int32_t* splat_count, uint32_t* zero_words,
                            int64_t n_zero_words, const float* depths,
                            void* depth_buffers, int walk,
                            hipStream_t stream, const CountHist& H) {
  if (P.num_splats == 0 || !depth_small_ok(P.gpb)) {
    set_error("count + depth runs: needs 1..131072 splats per image");
    return GSPLAT_ERR_INVALID_ARGUMENT;
  }
  const int runs = run_step::runs_of(P.gpb);
  const int run_blocks = P.batch * runs;
  const int cblocks = count_depth_runs_blocks(P, walk);
  launch_traced("count_depth_runs_kernel",
                walk == 8    ? count_depth_runs_kernel<8>
                : walk == 16 ? count_depth_runs_kernel<16>
                             : count_depth_runs_kernel<kWalkSplats>,
                dim3((unsigned)(run_blocks + cblocks)),
                dim3(run_step::kRunThreads), 0, stream, P, means2d, conics,
                opacities, splat_count, zero_words, n_zero_words, depths, runs,
                run_blocks,
                run_step::run_buffers(depth_buffers, P.gpb, P.batch), H);
  return check_launch("count_depth_runs_kernel");
}

int launch_rank_pack(const RasterParams& P, const float* means2d,
                     const float* conics, const float* colors,
                     const float* opacities, void* depth_buffers,
                     const int32_t* splat_count, int32_t* perm, float* packed,
                     int32_t* gid_count, uint32_t* block_totals, int walk,
                     hipStream_t stream, const CountHist& H) {
  if (P.num_splats == 0 || !depth_small_ok(P.gpb)) {
    set_error("rank + pack: needs 1..131072 splats per image");
    return GSPLAT_ERR_INVALID_ARGUMENT;
  }
  const int blocks_per_seg =
      (P.gpb + run_step::kRankElems - 1) / run_step::kRankElems;
  launch_traced("rank_pack_kernel", rank_pack_kernel,
                dim3((unsigned)((int64_t)P.batch * blocks_per_seg +
                                (H.parts != nullptr ? 1 : 0))),
                dim3(run_step::kRankBlock), 0, stream, P, means2d, conics,
                colors, opacities,
                run_step::run_buffers(depth_buffers, P.gpb, P.batch),
                run_step::runs_of(P.gpb), splat_count, perm,
                reinterpret_cast<float4*>(packed), gid_count, block_totals,
                kWaves * walk, H);
  return check_launch("rank_pack_kernel");
}

int launch_pack(const RasterParams& P, const float* means2d,
                const float* conics, const float* colors,
                const float* opacities, const uint32_t* perm,
                const int32_t* splat_count, float* packed,
                int32_t* splat_offsets, uint64_t* scan_status,
                uint32_t* scan_ticket, uint32_t* err, hipStream_t stream,
                const float* rec_orig, int32_t* orig_slot) {
  if (P.num_splats == 0) return GSPLAT_OK;
  const unsigned grid = (unsigned)((P.num_splats + kThreads - 1) / kThreads);
  launch_traced("pack_kernel", pack_kernel, dim3(grid), dim3(kThreads), 0,
                stream, P, means2d, conics, colors, opacities, perm,
                splat_count, reinterpret_cast<const float4*>(rec_orig),
                reinterpret_cast<float4*>(packed), splat_offsets, scan_status,
                scan_ticket, err, reinterpret_cast<int2*>(orig_slot));
  return check_launch("pack_kernel");
}

int launch_pack_records(const RasterParams& P, const float* means2d,
                        const float* conics, const float* colors,
                        const float* opacities, float* packed,
                        hipStream_t stream) {
  if (P.num_splats == 0) return GSPLAT_OK;
  const unsigned grid = (unsigned)((P.num_splats + kThreads - 1) / kThreads);
  launch_traced("pack_records_kernel", pack_records_kernel, dim3(grid),
                dim3(kThreads), 0, stream, P, means2d, conics, colors,
                opacities, reinterpret_cast<float4*>(packed));
  return check_launch("pack_records_kernel");
}

int count_scan_blocks(const RasterParams& P) {
  return (P.num_splats + kThreads - 1) / kThreads;
}

int emit_blocks(const RasterParams& P, int walk) {
  return (P.num_splats + kWaves * walk - 1) / (kWaves * walk);
}

int launch_emit(const RasterParams& P, const float* packed,
                const int32_t* splat_offsets, int64_t capacity, uint32_t* keys,
                uint32_t* vals, int pair_passes, uint32_t* hist_partials,
                uint32_t* pair_ghist, uint32_t* pair_status,
                int64_t pair_status_words, hipStream_t stream,
                const EmitScanArgs* scan, int hist_shift,
                uint8_t* key_bytes, const EmitOrigArgs* orig) {
  if (P.num_splats == 0) return GSPLAT_OK;
  const int nblk = emit_blocks(P, scan != nullptr ? scan->walk : kWalkSplats);
  // Few workgroups add their histograms atomically (pair_ghist is zeroed
  // by count_kernel), which saves the reduction launch; many would contend.
  const bool direct = nblk <= kDirectHistBlocks;
  if (scan != nullptr) {
    const EmitScan sc{scan->gid_count, scan->splat_offsets,
                      scan->block_totals};
    launch_traced("emit_kernel<true>",
                  scan->walk == 8    ? emit_kernel<true, false, 8>
                  : scan->walk == 16 ? emit_kernel<true, false, 16>
                                     : emit_kernel<true, false, kWalkSplats>,
                  dim3((unsigned)nblk), dim3(kThreads), 0, stream, P,
                  reinterpret_cast<const float4*>(packed), nullptr, capacity,
                  keys, vals, key_bytes, pair_passes, hist_shift, hist_partials,
                  direct ? pair_ghist : nullptr, pair_status, pair_status_words,
                  sc, EmitOrig{});
  } else if (orig != nullptr) {
    const EmitOrig eo{reinterpret_cast<const float4*>(orig->rec_orig),
                      reinterpret_cast<const int2*>(orig->orig_slot)};
    launch_traced("emit_kernel<orig>", emit_kernel<false, true, kWalkSplats>,
                  dim3((unsigned)nblk), dim3(kThreads), 0, stream, P,
                  reinterpret_cast<const float4*>(packed), splat_offsets,
                  capacity, keys, vals, key_bytes, pair_passes, hist_shift,
                  hist_partials,
                  direct ? pair_ghist : nullptr, pair_status, pair_status_words,
                  EmitScan{}, eo);
  } else {
    launch_traced("emit_kernel<false>", emit_kernel<false, false, kWalkSplats>,
                  dim3((unsigned)nblk), dim3(kThreads), 0, stream, P,
                  reinterpret_cast<const float4*>(packed), splat_offsets,
                  capacity, keys, vals, key_bytes, pair_passes, hist_shift,
                  hist_partials,
                  direct ? pair_ghist : nullptr, pair_status, pair_status_words,
                  EmitScan{}, EmitOrig{});
  }
  int rc = check_launch("emit_kernel");
  if (rc || pair_passes == 0 || direct) return rc;
  launch_traced("hist_reduce_kernel", hist_reduce_kernel,
                dim3((unsigned)(pair_passes * 256)), dim3(kThreads), 0, stream,
                hist_partials, nblk, pair_ghist);
  return check_launch("hist_reduce_kernel");
}

int launch_tile_ranges(const uint32_t* sorted_keys, int64_t n, int num_tiles,
                       int32_t* tile_offsets, int32_t* tile_counts,
                       hipStream_t stream, const int32_t* n_dev,
                       const uint32_t* err0, const uint32_t* err1,
                       const uint32_t* err2, int32_t* status_out,
                       int32_t* long_flag, const ZeroSpan* zero) {
  int rc = GSPLAT_OK;
  if (zero != nullptr && (num_tiles <= 0 || n == 0))
    rc = launch_zero2(zero[0].p, zero[0].n, zero[1].p, zero[1].n, stream);
  if (rc) return rc;
  if (num_tiles <= 0)
    return status_out ? launch_fill_i32(status_out, 0, 1, stream) : GSPLAT_OK;
  StatusWords sw{{err0, err1, err2}, status_out, long_flag, {}};
  if (zero != nullptr) {
    sw.zero[0] = zero[0];
    sw.zero[1] = zero[1];
  }
  if (n == 0) {
    rc = launch_fill_i32(tile_offsets, 0, (int64_t)num_tiles + 1, stream);
    if (!rc && status_out) rc = launch_fill_i32(status_out, 0, 1, stream);
  } else {
    int64_t grid = (n + 1 + kThreads - 1) / kThreads;
    if (grid > kRangeMaxBlocks) grid = kRangeMaxBlocks;
    launch_traced("ranges_kernel", ranges_kernel, dim3((unsigned)grid),
                  dim3(kThreads), 0, stream, sorted_keys, n, n_dev, num_tiles,
                  tile_offsets, sw);
    rc = check_launch("ranges_kernel");
  }
  if (rc || tile_counts == nullptr) return rc;
  launch_traced("counts_kernel", counts_kernel,
                dim3((unsigned)((num_tiles + kThreads - 1) / kThreads)),
                dim3(kThreads), 0, stream, tile_offsets, num_tiles,
                tile_counts);
  return check_launch("counts_kernel");
}

int launch_ranges_finish(int64_t n, int num_tiles, int32_t* tile_offsets,
                         int32_t* tile_counts, hipStream_t stream,
                         const int32_t* n_dev, const uint32_t* err0,
                         const uint32_t* err1, const uint32_t* err2,
                         int32_t* status_out, int32_t* long_flag,
                         const ZeroSpan* zero) {
  if (num_tiles <= 0 || n == 0)
    return launch_tile_ranges(nullptr, 0, num_tiles, tile_offsets, tile_counts,
                              stream, n_dev, err0, err1, err2, status_out,
                              long_flag, zero);
  StatusWords sw{{err0, err1, err2}, status_out, long_flag, {}};
  if (zero != nullptr) {
    sw.zero[0] = zero[0];
    sw.zero[1] = zero[1];
  }
  // (sized for the zero spans too)
  int64_t work = (int64_t)num_tiles + 1;
  for (int z = 0; z < 2; ++z) work = std::max(work, sw.zero[z].n);
  int64_t grid = (work + kThreads - 1) / kThreads;
  if (grid > kRangeMaxBlocks) grid = kRangeMaxBlocks;
  launch_traced("ranges_finish_kernel", ranges_finish_kernel,
                dim3((unsigned)grid), dim3(kThreads), 0, stream, n, n_dev,
                num_tiles, tile_offsets, sw);
  int rc = check_launch("ranges_finish_kernel");
  if (rc || tile_counts == nullptr) return rc;
  launch_traced("counts_kernel", counts_kernel,
                dim3((unsigned)((num_tiles + kThreads - 1) / kThreads)),
                dim3(kThreads), 0, stream, tile_offsets, num_tiles,
                tile_counts);
  return check_launch("counts_kernel");
}

int launch_bucket_sort(const BucketSortArgs& A, hipStream_t stream) {
  if (A.num_tiles <= 0 || A.low_bits < 1 || A.low_bits > 8) {
    set_error("bucket sort: needs tiles and 1..8 low bits");
    return GSPLAT_ERR_INVALID_ARGUMENT;
  }
  const int64_t buckets =
      ((int64_t)A.num_tiles + (1 << A.low_bits) - 1) >> A.low_bits;
  if (buckets > 256) {
    set_error("bucket sort: more than 256 buckets");
    return GSPLAT_ERR_INVALID_ARGUMENT;
  }
  launch_traced("bucket_sort_kernel", bucket_sort_kernel,
                dim3((unsigned)buckets), dim3(kBucketThreads), 0, stream, A);
  return check_launch("bucket_sort_kernel");
}

// Splats per wavefront: 16 up to 64K splats (a block per CU: count + emit at
// 64K splats 25.0 us at 1080p, 32.1 at 4096 x 4096, with 32 25.5 and 35.7), 32
// and 64 above (each emit block reads every block's counts: at most 256).
static int tile_walk(const RasterParams& P) {
  return P.num_splats <= (1 << 16) ? 16 : P.num_splats <= (1 << 17) ? 32 : 64;
}

int tile_blocks(const RasterParams& P) {
  const int splats = kTileWaves * tile_walk(P);
  return (P.num_splats + splats - 1) / splats;
}

int launch_tile_sorted(const RasterParams& P, const float* means2d,
                       const float* conics, const float* colors,
                       const float* opacities, const float* depths,
                       int low_bits, int64_t capacity, float* packed,
                       uint32_t* parts, uint32_t* bucket_start, int32_t* ctl,
                       void* pairs, int32_t* binned_ids, int32_t* tile_offsets,
                       int32_t* tile_ends, const ZeroSpan zero[2],
                       hipStream_t stream) {
  const unsigned blocks = (unsigned)tile_blocks(P);
  const int walk = tile_walk(P);
  launch_traced("tile_count_kernel",
                walk == 16   ? tile_count_kernel<16>
                : walk == 32 ? tile_count_kernel<32>
                             : tile_count_kernel<64>,
                dim3(blocks), dim3(kTileThreads), 0, stream, P, means2d,
                conics, colors, opacities, reinterpret_cast<float4*>(packed),
                parts, low_bits, ctl, zero[0], zero[1]);
  int rc = check_launch("tile_count_kernel");
  if (rc) return rc;
  launch_traced("tile_emit_kernel",
                walk == 16   ? tile_emit_kernel<16>
                : walk == 32 ? tile_emit_kernel<32>
                             : tile_emit_kernel<64>,
                dim3(blocks), dim3(kTileThreads), 0, stream, P, means2d,
                conics, opacities, depths, parts, low_bits, capacity,
                reinterpret_cast<uint2*>(pairs), bucket_start, ctl);
  rc = check_launch("tile_emit_kernel");
  if (rc) return rc;
  launch_traced("tile_sort_kernel", tile_sort_kernel,
                dim3((unsigned)(((int64_t)P.num_tiles + (1 << low_bits) - 1) >>
                                low_bits)),
                dim3(kTileThreads), 0, stream,
                reinterpret_cast<const uint2*>(pairs), bucket_start, capacity,
                P.num_tiles, low_bits,
                P.num_splats <= (1 << 16) ? kTileWorkSmall : kTileWork,
                reinterpret_cast<uint32_t*>(binned_ids), tile_offsets, tile_ends,
                ctl);
  return check_launch("tile_sort_kernel");
}

int launch_host_report(const HostReport& R, hipStream_t stream) {
  launch_traced("host_report_kernel", host_report_kernel, dim3(1), dim3(64), 0,
                stream, R);
  return check_launch("host_report_kernel");
}

int launch_zero2(uint32_t* a, int64_t na, uint32_t* b, int64_t nb,
                 hipStream_t stream) {
  const int64_t n = na > nb ? na : nb;
  if (n <= 0) return GSPLAT_OK;
  int64_t grid = (n + 255) / 256;
  if (grid > 4096) grid = 4096;
  launch_traced("zero2_kernel", zero2_kernel, dim3((unsigned)grid), dim3(256),
                0, stream, a, na, b, nb);
  return check_launch("zero2_kernel");
}

int launch_fill_i32(int32_t* dst, int32_t value, int64_t n,
                    hipStream_t stream) {
  if (n <= 0) return GSPLAT_OK;
  const int64_t grid = (n + 255) / 256;
  launch_traced("fill_i32_kernel", fill_i32_kernel, dim3((unsigned)grid),
                dim3(256), 0, stream, dst, value, n);
  return check_launch("fill_i32_kernel");
}

int launch_zero_grads(float* g_m, float* g_q, float* g_c, float* g_o,
                      int64_t n, hipStream_t stream) {
  if (n <= 0) return GSPLAT_OK;
  const int64_t grid = (3 * n + 255) / 256;
  launch_traced("zero_grads_kernel", zero_grads_kernel, dim3((unsigned)grid),
                dim3(256), 0, stream, g_m, g_q, g_c, g_o, n);
  return check_launch("zero_grads_kernel");
}

int launch_fill_f32(float* dst, float value, int64_t n, hipStream_t stream) {
  if (n <= 0) return GSPLAT_OK;
  const int64_t grid = (n + 255) / 256;
  launch_traced("fill_f32_kernel", fill_f32_kernel, dim3((unsigned)grid),
                dim3(256), 0, stream, dst, value, n);
  return check_launch("fill_f32_kernel");
}

}  // namespace gs
