// slice.hip -- the front slice of a dense scene: which splats it holds, which
// tiles it leaves live, and which splats those tiles still need.
//
// In a dense scene most of a tile's list lies behind the splat at which its
// last pixel became opaque: at 4096 x 4096 with 2^20 3D splats a tile lists
// 1862 pairs on average and walks 33 of them.  The sliced forward bins and
// composites the nearest splats alone (the front: as many as keep the pairs
// within a budget), finds the tiles where a pixel is still transparent (the
// live tiles), and bins all splats that touch a live tile, in live tiles
// only (the back); the live tiles are then composited again from their whole
// lists.  A tile that the front made opaque has walked a prefix of its list
// that holds its stop, so its image, stops and gradients are those of the
// whole list; a live tile's list is the whole one.  Both binnings are the
// ordinary ones, over compacted splats: what this file adds is the choice of
// the splats and of the tiles.
//
//   slice_hist_kernel<1>  each splat's tile box (kept), and per image the
//     counts of splats and of box tiles by the top 11 bits of the depth key
//   slice_hist_kernel<2>  the same by the next 11 bits, inside the bin where
//     the budget ends (slice_limit_kernel<1>)
//   slice_limit_kernel<2> the 22-bit key where it ends
//   slice_front_kernel    compacts the splats before that 22-bit key, in
//     original order (stable depth ties), with their attributes
//   slice_live_kernel     the live tiles as a bitmap and a list
//   slice_select_kernel   compacts the splats whose box holds a live tile, cuts
//     their boxes down to those tiles and sums the live tiles in them (a
//     bound on the back's pairs)
//   slice_report_kernel   what the host needs to launch the back, and a stop of
//     0 for the live tiles if there is one
//   slice_gather_kernel   the back's attributes, once the host knows its size
//
// The budget counts box tiles, at least the pairs the binning emits, so the
// buffers of a slice never overflow.  The histograms and the front read each
// splat once (18 to 38 MB at 2^20 splats) in 16 to 18 us, 1.0 to 2.2 TB/s where
// a large copy reaches 4.9: launch and load latency; the selection (45 us, 10
// MB, vector units busy for 38%) is bound by its walk over the boxes' rows.
#include <algorithm>

#include "gs_internal.h"
#include "gs_predicate.h"
#include "lookback.h"

namespace gs {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
// Splats per thread: the histograms' workgroups take more (each clears and
// adds 2048 bins), the compactions' fewer (a box of many tile rows keeps its
// lane for long, and 100K splats should fill the chip).
constexpr int kHistRounds = 8;
constexpr int kRounds = 4;
constexpr int kBins = 2048;
constexpr int kBinsPerThread = kBins / kThreads;
// A histogram word: box tiles, and splats above them (one atomic for both).
// (Fewer than 2^22 splats of at most 2^18 tiles: slice_ok.)
constexpr int kCountShift = 40;

int blocks_per_image(const RasterParams& P, int rounds) {
  return (P.gpb + kThreads * rounds - 1) / (kThreads * rounds);
}

// Index inside the image of round r of this thread's splats: blocks,
// wavefronts, rounds and lanes ascend in this order.
template <int kN>
__device__ __forceinline__ int splat_in_image(int blk, int r) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  return (blk * kWaves + wave) * 64 * kN + 64 * r + lane;
}

// The tile box of a splat, the candidates of the binning's walk: corner and
// size in tiles, 16 bits each; no tiles: 0.
__device__ __forceinline__ uint2 tile_box(const RasterParams& P,
                                          const float* __restrict__ means2d,
                                          const float* __restrict__ conics,
                                          const float* __restrict__ opacities,
                                          int64_t i) {
  float tau;
  if (!alpha_support(opacities[i], P.alpha_thr, P.eps, tau))
    return make_uint2(0u, 0u);
  const PixBox b = snugbox(means2d[2 * i], means2d[2 * i + 1], conics[3 * i],
                           conics[3 * i + 1], conics[3 * i + 2], tau, P.width,
                           P.height, P.eps);
  if (!(b.x0 <= b.x1 && b.y0 <= b.y1)) return make_uint2(0u, 0u);
  const uint32_t tx0 = (uint32_t)(b.x0 >> 4), ty0 = (uint32_t)(b.y0 >> 4);
  const uint32_t w = (uint32_t)(b.x1 >> 4) - tx0 + 1u;
  const uint32_t h = (uint32_t)(b.y1 >> 4) - ty0 + 1u;
  return make_uint2(tx0 | ty0 << 16, w | h << 16);
}
__device__ __forceinline__ uint32_t box_tiles(uint2 b) {
  return (b.y & 0xffffu) * (b.y >> 16);
}

// Exclusive scan of (c, t) over the workgroup's threads, and the totals.
struct ScanLds {
  unsigned long long c[kWaves], t[kWaves];
  int bin;
  uint32_t at_c;
  unsigned long long at_t;
};
__device__ __forceinline__ void block_scan(unsigned long long& c,
                                           unsigned long long& t, ScanLds& S,
                                           unsigned long long& all_c,
                                           unsigned long long& all_t) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long c0 = c, t0 = t;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned long long yc = __shfl_up(c, off, 64);
    const unsigned long long yt = __shfl_up(t, off, 64);
    if (lane >= off) {
      c += yc;
      t += yt;
    }
  }
  if (lane == 63) {
    S.c[wave] = c;
    S.t[wave] = t;
  }
  __syncthreads();
  unsigned long long pc = 0, pt = 0;
  all_c = all_t = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    pc += w < wave ? S.c[w] : 0ull;
    pt += w < wave ? S.t[w] : 0ull;
    all_c += S.c[w];
    all_t += S.t[w];
  }
  c = pc + c - c0;
  t = pt + t - t0;
  __syncthreads();
}

// The first bin that would take the running totals (from c0, t0) above
// max_c splats or max_t tiles, kBins if none does, and the totals before it.
__device__ __forceinline__ SliceCrossing find_crossing(
    const unsigned long long* __restrict__ hist, uint32_t c0,
    unsigned long long t0, uint32_t max_c, unsigned long long max_t,
    ScanLds& S, unsigned long long& all_t) {
  const int b0 = (int)threadIdx.x * kBinsPerThread;
  uint32_t bc[kBinsPerThread];
  unsigned long long bt[kBinsPerThread], c = 0, t = 0, all_c;
#pragma unroll
  for (int k = 0; k < kBinsPerThread; ++k) {
    const unsigned long long v = hist[b0 + k];
    bc[k] = (uint32_t)(v >> kCountShift);
    bt[k] = v & ((1ull << kCountShift) - 1ull);
    c += bc[k];
    t += bt[k];
  }
  if (threadIdx.x == 0) S.bin = kBins;
  block_scan(c, t, S, all_c, all_t);  // (synchronises: S.bin is set)
  c += c0;
  t += t0;
  int bin = kBins;
  uint32_t at_c = 0;
  unsigned long long at_t = 0;
#pragma unroll
  for (int k = 0; k < kBinsPerThread; ++k) {
    if (bin == kBins && (c + bc[k] > max_c || t + bt[k] > max_t)) {
      bin = b0 + k;
      at_c = (uint32_t)c;
      at_t = t;
    }
    c += bc[k];
    t += bt[k];
  }
  if (bin < kBins) atomicMin(&S.bin, bin);
  __syncthreads();
  const int first = S.bin;
  if (first < kBins && bin == first) {
    S.at_c = at_c;
    S.at_t = at_t;
  }
  __syncthreads();
  SliceCrossing r;
  r.bin = first;
  r.c = first < kBins ? S.at_c : (uint32_t)(c0 + all_c);
  r.t = first < kBins ? S.at_t : t0 + all_t;
  __syncthreads();  // S is used again
  return r;
}

// One workgroup per image: where the budget ends at this level (a kernel of
// its own: found by every workgroup of the next one it cost each of those
// about 10 us).
template <int kLevel>
__global__ __launch_bounds__(kThreads) void slice_limit_kernel(
    RasterParams P, SliceBuffers Q, int slots, long long max_tiles) {
  __shared__ ScanLds S;
  const int img = (int)blockIdx.x;
  const int64_t row = (int64_t)(kLevel == 1 ? img : P.batch + img) * kBins;
  const SliceCrossing c1 = kLevel == 1 ? SliceCrossing{} : Q.cross[img];
  unsigned long long all;
  const SliceCrossing c =
      find_crossing(Q.hist + row, c1.c, c1.t, (uint32_t)slots,
                    (unsigned long long)max_tiles, S, all);
  if (threadIdx.x != 0) return;
  if (kLevel == 1) {
    Q.cross[img] = c;
    atomicAdd(&Q.sums[kSliceTilesAll], all);
  } else if (c1.bin >= kBins) {
    Q.limit[img] = (uint32_t)kBins << 11;  // every splat
  } else {
    // (the bin's totals went above the budget, so a bin crosses here)
    Q.limit[img] = ((uint32_t)c1.bin << 11) + (uint32_t)c.bin;
  }
}

template <int kLevel>
__global__ __launch_bounds__(kThreads) void slice_hist_kernel(
    RasterParams P, SliceBuffers Q, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ opacities,
    const float* __restrict__ depths, int slots) {
  __shared__ uint32_t cnt[kBins], tiles[kBins];
  const int img = (int)blockIdx.y, t = threadIdx.x;
  for (int i = t; i < kBins; i += kThreads) cnt[i] = tiles[i] = 0u;
  int only = 0;
  if (kLevel == 2) {
    only = Q.cross[img].bin;
    // the front's slots start as padding: splats without tiles, last in
    // depth order
    const int64_t n = (int64_t)slots * P.batch;
    for (int64_t i = ((int64_t)img * gridDim.x + blockIdx.x) * kThreads + t;
         i < n; i += (int64_t)gridDim.x * gridDim.y * kThreads) {
      Q.front.opacities[i] = 0.0f;
      Q.front.depths[i] = __builtin_inff();
      Q.front.orig[i] = 0;
    }
  }
  __syncthreads();
  // (level 2: all loads in flight before the first use)
  uint32_t key[kHistRounds];
  uint2 box[kHistRounds];
#pragma unroll
  for (int r = 0; r < kHistRounds; ++r) {
    const int e = splat_in_image<kHistRounds>((int)blockIdx.x, r);
    const int64_t i = (int64_t)img * P.gpb + min(e, P.gpb - 1);
    key[r] = depth_key(depths[i]);
    if (kLevel == 2) box[r] = Q.box[i];
  }
#pragma unroll
  for (int r = 0; r < kHistRounds; ++r) {
    const int e = splat_in_image<kHistRounds>((int)blockIdx.x, r);
    const int64_t i = (int64_t)img * P.gpb + min(e, P.gpb - 1);
    if (kLevel == 1) {
      box[r] = tile_box(P, means2d, conics, opacities, i);
      if (e < P.gpb) Q.box[i] = box[r];
    }
    const uint32_t n = e < P.gpb ? box_tiles(box[r]) : 0u;
    if (n == 0u || (kLevel == 2 && (int)(key[r] >> 21) != only)) continue;
    const uint32_t bin =
        kLevel == 1 ? key[r] >> 21 : (key[r] >> 10) & (uint32_t)(kBins - 1);
    atomicAdd(&cnt[bin], 1u);
    atomicAdd(&tiles[bin], n);  // (2048 boxes of at most 2^18 tiles)
  }
  __syncthreads();
  const int64_t row = (int64_t)(kLevel == 1 ? img : P.batch + img) * kBins;
  for (int i = t; i < kBins; i += kThreads)
    if (cnt[i] != 0u) {
      atomicAdd(&Q.hist[row + i], (unsigned long long)tiles[i] |
                                      (unsigned long long)cnt[i] << kCountShift);
    }
}

// Order-keeping compaction of a block's flagged splats (m[r]: the
// wavefront's ballot of round r): the image's splats flagged before this
// block by a look-back over its blocks (status: the image's row), then the
// wavefronts' totals.  Blocks go by workgroup index, not by a ticket, as in
// the pair sort's passes (radix_sort.hip): 2048 atomics on one word held the
// launch for 20 us.  Returns the position of this wavefront's first
// flagged splat; total: those of the block.
__device__ __forceinline__ uint32_t compact_base(const uint64_t (&m)[kRounds],
                                                 uint64_t* status, int blk,
                                                 uint32_t* err, uint32_t* wsum,
                                                 uint32_t* s_prefix,
                                                 uint32_t& end) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t n = 0u;
#pragma unroll
  for (int r = 0; r < kRounds; ++r) n += (uint32_t)__popcll(m[r]);
  if (lane == 0) wsum[wave] = n;
  __syncthreads();
  uint32_t pre = 0u, total = 0u;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    pre += w < wave ? wsum[w] : 0u;
    total += wsum[w];
  }
  if (wave == 0) {
    if (lane == 0)
      status_store(&status[blk], (blk == 0 ? kFlagInc64 : kFlagAgg64) | total);
    uint64_t prefix = 0ull;
    if (blk > 0) {
      prefix = lookback64_wave(status, blk, err);
      if (lane == 0) status_store(&status[blk], kFlagInc64 | (prefix + total));
    }
    if (lane == 0) *s_prefix = (uint32_t)prefix;
  }
  __syncthreads();
  end = *s_prefix + total;
  return *s_prefix + pre;
}

__device__ __forceinline__ void copy_splat(const SliceSplats& D, int64_t to,
                                           const float* __restrict__ means2d,
                                           const float* __restrict__ conics,
                                           const float* __restrict__ colors,
                                           const float* __restrict__ opacities,
                                           const float* __restrict__ depths,
                                           int64_t i) {
  D.means2d[2 * to] = means2d[2 * i];
  D.means2d[2 * to + 1] = means2d[2 * i + 1];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    D.conics[3 * to + k] = conics[3 * i + k];
    D.colors[3 * to + k] = colors[3 * i + k];
  }
  D.opacities[to] = opacities[i];
  D.depths[to] = depths[i];
  D.orig[to] = (int32_t)i;
}

__global__ __launch_bounds__(kThreads) void slice_front_kernel(
    RasterParams P, SliceBuffers Q, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ colors,
    const float* __restrict__ opacities, const float* __restrict__ depths,
    int slots, int blocks) {
  __shared__ uint32_t wsum[kWaves];
  __shared__ uint32_t s_prefix;
  const int vb = (int)blockIdx.x;
  const int img = vb / blocks, blk = vb - img * blocks;
  const uint32_t limit = Q.limit[img];
  const int lane = threadIdx.x & 63;
  uint64_t m[kRounds];
  uint32_t key[kRounds], size[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int e = splat_in_image<kRounds>(blk, r);
    const int64_t i = (int64_t)img * P.gpb + min(e, P.gpb - 1);
    key[r] = depth_key(depths[i]);
    size[r] = e < P.gpb ? Q.box[i].y : 0u;
  }
#pragma unroll
  for (int r = 0; r < kRounds; ++r)
    m[r] = __ballot((key[r] >> 10) < limit && size[r] != 0u);
  uint32_t end;
  uint32_t pos = compact_base(m, Q.status_front + (int64_t)img * blocks, blk,
                              &Q.ctl[kSliceErr], wsum, &s_prefix, end);
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const uint32_t p = pos + (uint32_t)__popcll(m[r] & ((1ull << lane) - 1ull));
    pos += (uint32_t)__popcll(m[r]);
    // (p < slots by the choice of the limit; a look-back that gave up must
    // not leave the buffers)
    if (((m[r] >> lane) & 1ull) != 0ull && p < (uint32_t)slots)
      copy_splat(Q.front, (int64_t)img * slots + p, means2d, conics, colors,
                 opacities, depths,
                 (int64_t)img * P.gpb + splat_in_image<kRounds>(blk, r));
  }
}

// 1024 tiles per workgroup: the live tiles' bits and their list (ascending
// inside a workgroup).  Also the sum and number of the opaque tiles' stops.
__global__ __launch_bounds__(kThreads) void slice_live_kernel(
    RasterParams P, SliceBuffers Q, const uint32_t* __restrict__ tile_live,
    const int32_t* __restrict__ tile_stop) {
  __shared__ uint32_t wsum[kWaves];
  __shared__ uint32_t s_base;
  __shared__ uint32_t s_stops, s_opaque;
  if (threadIdx.x == 0) s_stops = s_opaque = 0u;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t0 = (int)blockIdx.x * (4 * kThreads) + wave * 256;
  uint64_t m[4];
  uint32_t n = 0u, stops = 0u, opaque_n = 0u;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = t0 + 64 * r + lane;
    const bool in = t < P.num_tiles;
    const bool live = in && tile_live[min(t, P.num_tiles - 1)] != 0u;
    m[r] = __ballot(live);
    n += (uint32_t)__popcll(m[r]);
    if (lane < 2 && t0 + 64 * r + 32 * lane < P.num_tiles)
      Q.live_bits[(t0 + 64 * r) / 32 + lane] = (uint32_t)(m[r] >> (32 * lane));
    if (in && !live) {
      stops += (uint32_t)tile_stop[t];
      ++opaque_n;
    }
  }
  if (lane == 0) wsum[wave] = n;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    stops += __shfl_xor(stops, off, 64);
    opaque_n += __shfl_xor(opaque_n, off, 64);
  }
  if (lane == 0) {  // (a stop is below 2^20: the front's slots per image)
    atomicAdd(&s_stops, stops);
    atomicAdd(&s_opaque, opaque_n);
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_opaque != 0u) {
    atomicAdd(&Q.sums[kSliceStops], (unsigned long long)s_stops);
    atomicAdd(&Q.sums[kSliceOpaque], (unsigned long long)s_opaque);
  }
  uint32_t pre = 0u, total = 0u;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    pre += w < wave ? wsum[w] : 0u;
    total += wsum[w];
  }
  if (threadIdx.x == 0)
    s_base = total != 0u ? atomicAdd(&Q.ctl[kSliceLive], total) : 0u;
  __syncthreads();
  uint32_t pos = s_base + pre;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (((m[r] >> lane) & 1ull) != 0ull)
      Q.live_list[pos + (uint32_t)__popcll(m[r] & ((1ull << lane) - 1ull))] =
          t0 + 64 * r + lane;
    pos += (uint32_t)__popcll(m[r]);
  }
}

// The rows of 64 splats' boxes, 64 at a time whatever splats they belong to
// (a lane per splat would hold its wavefront for the tallest box: 77 us
// instead of 44 at 2^20 splats of which a tenth have boxes of up to 70 rows).
struct SelectLds {
  int end[64];       // inclusive prefix sum of the splats' rows
  uint32_t live[64]; // live tiles of the box
  uint32_t x0[64], x1[64], y0[64], y1[64];  // their extent
};

__global__ __launch_bounds__(kThreads) void slice_select_kernel(
    RasterParams P, SliceBuffers Q, const float* __restrict__ depths,
    int blocks, int lds_words) {
  extern __shared__ uint32_t bits[];  // the image's live bits
  __shared__ SelectLds lds[kWaves];
  __shared__ uint32_t wsum[kWaves];
  __shared__ uint32_t s_prefix;
  __shared__ unsigned long long s_tiles;
  __shared__ uint32_t s_new;
  const int vb = (int)blockIdx.x;
  const int img = vb / blocks, blk = vb - img * blocks;
  const int lane = threadIdx.x & 63;
  SelectLds& W = lds[threadIdx.x >> 6];
  const uint32_t limit = Q.limit[img];
  const int first_bit = img * P.tiles_per_image;
  const int first_word = first_bit >> 5;
  const int words = ((first_bit + P.tiles_per_image - 1) >> 5) - first_word + 1;
  for (int i = threadIdx.x; i < words && i < lds_words; i += kThreads)
    bits[i] = Q.live_bits[first_word + i];
  if (threadIdx.x == 0) {
    s_tiles = 0ull;
    s_new = 0u;
  }
  __syncthreads();
  uint64_t m[kRounds];
  uint32_t fresh = 0u;
  unsigned long long sum = 0ull;
#pragma unroll 1
  for (int r = 0; r < kRounds; ++r) {
    const int e = splat_in_image<kRounds>(blk, r);
    const int64_t i = (int64_t)img * P.gpb + min(e, P.gpb - 1);
    const uint2 b = e < P.gpb ? Q.box[i] : make_uint2(0u, 0u);
    int inc = (int)(b.y >> 16);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(inc, off, 64);
      if (lane >= off) inc += y;
    }
    W.end[lane] = inc;
    W.live[lane] = W.x1[lane] = W.y1[lane] = 0u;
    W.x0[lane] = W.y0[lane] = ~0u;
    const int rows = __shfl(inc, 63, 64);
    // (one wavefront: its LDS accesses take effect in program order)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int k0 = 0; k0 < rows; k0 += 64) {
      const int k = k0 + lane;
      // the row's splat: the number of splats that end at or before it
      int s = 0;
#pragma unroll
      for (int step = 32; step > 0; step >>= 1)
        if (W.end[s + step - 1] <= k) s += step;
      s = min(s, 63);
      const uint32_t bx = (uint32_t)__shfl((int)b.x, s, 64);
      const uint32_t by = (uint32_t)__shfl((int)b.y, s, 64);
      const int w = (int)(by & 0xffffu), h = (int)(by >> 16);
      if (k < rows) {
        const int ty = (int)(bx >> 16) + k - (W.end[s] - h);
        const int tx0 = (int)(bx & 0xffffu);
        const int bit = first_bit - 32 * first_word + ty * P.tiles_x + tx0;
        const int last = bit + w - 1;
        uint32_t n = 0u;
        int lo = 0, hi = 0;
        for (int q = bit >> 5; q <= (last >> 5); ++q) {
          uint32_t v = bits[q];
          if (q == (bit >> 5)) v &= ~0u << (bit & 31);
          if (q == (last >> 5)) v &= ~0u >> (31 - (last & 31));
          if (v != 0u) {
            if (n == 0u) lo = 32 * q + __ffs((int)v) - 1;
            hi = 32 * q + 31 - __clz((int)v);
            n += (uint32_t)__popc(v);
          }
        }
        if (n != 0u) {
          atomicAdd(&W.live[s], n);
          atomicMin(&W.x0[s], (uint32_t)(tx0 + lo - bit));
          atomicMax(&W.x1[s], (uint32_t)(tx0 + hi - bit));
          atomicMin(&W.y0[s], (uint32_t)ty);
          atomicMax(&W.y1[s], (uint32_t)ty);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t n = W.live[lane];
    if (n != 0u) {
      Q.box[i] = make_uint2(W.x0[lane] | W.y0[lane] << 16,
                            (W.x1[lane] - W.x0[lane] + 1u) |
                                (W.y1[lane] - W.y0[lane] + 1u) << 16);
      if ((depth_key(depths[i]) >> 10) >= limit) fresh = 1u;
    }
    sum += n;
    m[r] = __ballot(n != 0u);
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off, 64);
    fresh |= __shfl_xor(fresh, off, 64);
  }
  if (lane == 0) {
    atomicAdd(&s_tiles, sum);
    atomicOr(&s_new, fresh);
  }
  uint32_t end;
  uint32_t pos = compact_base(m, Q.status_back + (int64_t)img * blocks, blk,
                              &Q.ctl[kSliceErr], wsum, &s_prefix, end);
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const uint32_t p = pos + (uint32_t)__popcll(m[r] & ((1ull << lane) - 1ull));
    pos += (uint32_t)__popcll(m[r]);
    if (((m[r] >> lane) & 1ull) != 0ull && p < (uint32_t)P.gpb)
      Q.back_list[(int64_t)img * P.gpb + p] =
          img * P.gpb + splat_in_image<kRounds>(blk, r);
  }
  if (threadIdx.x == 0) {
    if (s_tiles != 0ull) atomicAdd(&Q.sums[kSliceTilesBack], s_tiles);
    if (s_new != 0u) atomicOr(&Q.ctl[kSliceFresh], 1u);
    if (blk == blocks - 1) {
      Q.back_count[img] = min(end, (uint32_t)P.gpb);
      atomicMax(&Q.ctl[kSliceBackMax], min(end, (uint32_t)P.gpb));
    }
  }
}

// What the host reads (the words of gsplat_hip_front_render), the ready word
// last; and, if a live tile needs splats that the front does not hold, a stop
// of 0 for the live tiles, so that the front's backward leaves them to the
// back's.  Without such a splat there is no back (the host goes by the same
// word), and the front's stops stand.
__global__ __launch_bounds__(kThreads) void slice_report_kernel(
    RasterParams P, SliceBuffers Q, const uint32_t* __restrict__ tile_live,
    int32_t* __restrict__ tile_stop, const int32_t* __restrict__ bin_status,
    int32_t* host) {
  const uint32_t fresh = Q.ctl[kSliceFresh];
  if (fresh != 0u) {
    for (int t = (int)blockIdx.x * kThreads + (int)threadIdx.x;
         t < P.num_tiles; t += (int)gridDim.x * kThreads)
      if (tile_live[t] != 0u) tile_stop[t] = 0;
  }
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  auto put = [&](int k, uint32_t v) {
    __hip_atomic_store(host + k, (int32_t)v, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  };
  put(0, (uint32_t)*bin_status | Q.ctl[kSliceErr]);
  put(1, Q.ctl[kSliceLive]);
  put(2, Q.ctl[kSliceBackMax]);
  put(3, fresh);
#pragma unroll
  for (int k = 0; k < kSliceSums; ++k) {
    put(4 + 2 * k, (uint32_t)Q.sums[k]);
    put(5 + 2 * k, (uint32_t)(Q.sums[k] >> 32));
  }
  __hip_atomic_store(host + 15, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ __launch_bounds__(kThreads) void slice_gather_kernel(
    RasterParams P, SliceBuffers Q, SliceSplats D, int slots,
    const float* __restrict__ means2d, const float* __restrict__ conics,
    const float* __restrict__ colors, const float* __restrict__ opacities,
    const float* __restrict__ depths) {
  const int img = (int)blockIdx.y;
  const int p = (int)blockIdx.x * kThreads + (int)threadIdx.x;
  if (p >= slots) return;
  const int64_t to = (int64_t)img * slots + p;
  if (p < (int)Q.back_count[img]) {
    // (the list is written up to the count unless a look-back gave up)
    const int32_t i = min(max(Q.back_list[(int64_t)img * P.gpb + p], 0),
                          P.num_splats - 1);
    copy_splat(D, to, means2d, conics, colors, opacities, depths, i);
  } else {
    D.opacities[to] = 0.0f;
    D.depths[to] = __builtin_inff();
    D.orig[to] = 0;
  }
}

}  // namespace

// Per image fewer than 2^22 splats (kCountShift: 2^22 boxes of 2^18 tiles)
// and at most 2^18 tiles (the select kernel keeps an image's live bits
// in LDS, and a block's 2048 boxes of that many tiles fit 32-bit sums) and
// 2^16 - 1 tiles a side (16-bit boxes).  The slots left over hold opacity 0,
// which is without tiles only at a threshold of 0 or more.
bool slice_ok(const RasterParams& P) {
  return P.num_tiles > 0 && P.num_splats > 0 && P.batch <= 64 &&
         P.gpb < (1 << 22) && P.alpha_thr >= 0.0f &&
         P.tiles_per_image <= (1 << 18) && P.tiles_x < (1 << 16) &&
         P.tiles_y < (1 << 16);
}

int slice_status_words(const RasterParams& P) {
  return P.batch * blocks_per_image(P, kRounds);
}

int launch_slice_front(const RasterParams& P, const SliceBuffers& Q,
                       const float* means2d, const float* conics,
                       const float* colors, const float* opacities,
                       const float* depths, int slots, int64_t max_tiles,
                       hipStream_t stream) {
  const int blocks = blocks_per_image(P, kRounds);
  const dim3 grid((unsigned)blocks_per_image(P, kHistRounds), (unsigned)P.batch);
  launch_traced("slice_hist_kernel<1>", slice_hist_kernel<1>, grid,
                dim3(kThreads), 0, stream, P, Q, means2d, conics, opacities,
                depths, slots);
  int rc = check_launch("slice_hist_kernel");
  if (rc) return rc;
  launch_traced("slice_limit_kernel<1>", slice_limit_kernel<1>,
                dim3((unsigned)P.batch), dim3(kThreads), 0, stream, P, Q,
                slots, (long long)max_tiles);
  rc = check_launch("slice_limit_kernel");
  if (rc) return rc;
  launch_traced("slice_hist_kernel<2>", slice_hist_kernel<2>, grid,
                dim3(kThreads), 0, stream, P, Q, means2d, conics, opacities,
                depths, slots);
  rc = check_launch("slice_hist_kernel");
  if (rc) return rc;
  launch_traced("slice_limit_kernel<2>", slice_limit_kernel<2>,
                dim3((unsigned)P.batch), dim3(kThreads), 0, stream, P, Q,
                slots, (long long)max_tiles);
  rc = check_launch("slice_limit_kernel");
  if (rc) return rc;
  launch_traced("slice_front_kernel", slice_front_kernel,
                dim3((unsigned)(blocks * P.batch)), dim3(kThreads), 0, stream,
                P, Q, means2d, conics, colors, opacities, depths, slots,
                blocks);
  return check_launch("slice_front_kernel");
}

int launch_slice_back(const RasterParams& P, const SliceBuffers& Q,
                      const float* depths, const uint32_t* tile_live,
                      int32_t* tile_stop, const int32_t* bin_status,
                      int32_t* host_words, hipStream_t stream) {
  launch_traced("slice_live_kernel", slice_live_kernel,
                dim3((unsigned)((P.num_tiles + 4 * kThreads - 1) / (4 * kThreads))),
                dim3(kThreads), 0, stream, P, Q, tile_live, tile_stop);
  int rc = check_launch("slice_live_kernel");
  if (rc) return rc;
  const int blocks = blocks_per_image(P, kRounds);
  const int words = (P.tiles_per_image + 31) / 32 + 1;
  launch_traced("slice_select_kernel", slice_select_kernel,
                dim3((unsigned)(blocks * P.batch)), dim3(kThreads),
                (size_t)words * sizeof(uint32_t), stream, P, Q, depths, blocks,
                words);
  rc = check_launch("slice_select_kernel");
  if (rc) return rc;
  launch_traced("slice_report_kernel", slice_report_kernel,
                dim3((unsigned)std::min((P.num_tiles + kThreads - 1) / kThreads,
                                        256)),
                dim3(kThreads), 0, stream, P, Q, tile_live, tile_stop,
                bin_status, host_words);
  return check_launch("slice_report_kernel");
}

int launch_slice_gather(const RasterParams& P, const SliceBuffers& Q,
                        const SliceSplats& to, int slots, const float* means2d,
                        const float* conics, const float* colors,
                        const float* opacities, const float* depths,
                        hipStream_t stream) {
  launch_traced("slice_gather_kernel", slice_gather_kernel,
                dim3((unsigned)((slots + kThreads - 1) / kThreads),
                     (unsigned)P.batch),
                dim3(kThreads), 0, stream, P, Q, to, slots, means2d, conics,
                colors, opacities, depths);
  return check_launch("slice_gather_kernel");
}

}  // namespace gs
