// direct.hip -- the binning of small scenes: every tile scans its image's
// splats.
//
// A few hundred to a few thousand splats on a few hundred tiles take the
// one-call binning five launches (run sort, ranks, emit and two sort steps,
// 40 to 50 us, nearly all of it launch latency and serial chains) and the
// host a wait for the pair count.  Here one launch ranks and packs the
// splats, and a second has each tile test the image's splats in depth order
// and write its list, in place for the compositors: G entries are kept per
// tile, so no count is needed beforehand and nothing can overflow.
//
// direct_pack_kernel  16 threads a splat count the keys before its own (LDS,
//   two VALU operations a key): 5 us at 300 splats, 18 at 5 x 4001, where the
//   80M compares bound it (one key a read and a four-operation test: 27).
// direct_list_kernel  a wavefront per tile: 64 tile boxes a step, the splats
//   whose box holds the tile compacted in LDS, then tested exactly 64 at a
//   time.  Bound by the tiles x splats box tests: 4.5 us at 1024 tiles x
//   512 splats, 14 at 1430 x 4001.
// Both together: 512 splats at 512 x 512 41 -> 10 us, five images of 4001
// splats 46 -> 33 us, and the forward's caller no longer waits.
//
// Compiled with -ffp-contract=off, like binning.hip: the lists are those of
// the other paths bit for bit.
#include <algorithm>

#include "gs_internal.h"
#include "record.h"

namespace gs {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
// The rank kernel: 64 splats a workgroup (one wavefront packs them), 16
// threads a splat, four keys a read.
constexpr int kPackThreads = 1024;
constexpr int kPackSplats = 64;
constexpr int kRankSplit = kPackThreads / kPackSplats;
constexpr int kBoxUnroll = 8;  // box loads in flight per lane

__global__ __launch_bounds__(kPackThreads) void direct_pack_kernel(
    RasterParams P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ colors,
    const float* __restrict__ opacities, const float* __restrict__ depths,
    float4* __restrict__ packed, DirectSplats D, ZeroSpan z0, ZeroSpan z1) {
  __shared__ uint4 key4[kDirectMaxSplats / 4];
  __shared__ int ranks[kPackSplats];
  uint32_t* key = reinterpret_cast<uint32_t*>(key4);
  const int t = threadIdx.x, img = (int)blockIdx.y, G = P.gpb;
  const int64_t base = (int64_t)img * G;
  const int64_t first =
      ((int64_t)img * gridDim.x + blockIdx.x) * kPackThreads + t;
  const int64_t stride = (int64_t)gridDim.x * gridDim.y * kPackThreads;
  for (int64_t i = first; i < z0.n; i += stride) z0.p[i] = 0u;
  for (int64_t i = first; i < z1.n; i += stride) z1.p[i] = 0u;
  // (the last word of four is filled up with keys above every depth's)
  const int G4 = (G + 3) / 4;
  for (int j = t; j < 4 * G4; j += kPackThreads)
    key[j] = j < G ? depth_key(depths[base + j]) : 0xffffffffu;
  __syncthreads();
  // stable rank: smaller keys, and equal ones of smaller index
  const int i0 = (int)blockIdx.x * kPackSplats;
  {
    const int i = i0 + t / kRankSplit;
    const uint32_t ki = key[min(i, G - 1)];
    int rank = 0;
    // words of four before the splat's own count keys <= ki, as < ki + 1 (no
    // depth key is 2^32 - 1); the others keys < ki, and the equal ones
    // before the splat in its own word are added below
    const int own = i >> 2;
#pragma unroll 4
    for (int q = t % kRankSplit; q < G4; q += kRankSplit) {
      const uint4 k = key4[q];
      const uint32_t lim = ki + (uint32_t)(q < own);
      rank += (int)(k.x < lim);
      rank += (int)(k.y < lim);
      rank += (int)(k.z < lim);
      rank += (int)(k.w < lim);
    }
    if (t % kRankSplit < 3 && 4 * own + t % kRankSplit < i && i < G)
      rank += (int)(key[4 * own + t % kRankSplit] == ki);
#pragma unroll
    for (int off = kRankSplit / 2; off > 0; off >>= 1)
      rank += __shfl_xor(rank, off, 64);
    if (t % kRankSplit == 0) ranks[t / kRankSplit] = rank;
  }
  __syncthreads();
  const int i = i0 + t;
  if (t >= kPackSplats || i >= G) return;
  const int rank = ranks[t];
  const int64_t orig = base + i, gid = base + rank;
  const Record r = record_of(P, means2d, conics, colors, opacities, (int)orig,
                             (uint32_t)orig);
  store_record(packed, gid, r);
  // inclusive tile box {x0 | y0 << 16, x1 | y1 << 16}; no tiles: x0 > x1
  uint2 box = make_uint2(0xffffu, 0u);
  float tau = 0.0f;
  const float a = r.v[0].z, b = r.v[0].w, c = r.v[1].x;
  if (alpha_support(r.v[1].y, P.alpha_thr, P.eps, tau)) {
    const PixBox q =
        snugbox(r.v[0].x, r.v[0].y, a, b, c, tau, P.width, P.height, P.eps);
    if (q.x0 <= q.x1 && q.y0 <= q.y1)
      box = make_uint2((uint32_t)(q.x0 >> 4) | (uint32_t)(q.y0 >> 4) << 16,
                       (uint32_t)(q.x1 >> 4) | (uint32_t)(q.y1 >> 4) << 16);
  }
  const ConicSlopes k = conic_slopes(a, b, c);
  D.box[gid] = box;
  D.test[gid] = make_float4(
      tau, k.kc, k.ka,
      __uint_as_float((k.use_c ? 1u : 0u) | (k.use_a ? 2u : 0u)));
}

__global__ __launch_bounds__(kThreads) void direct_list_kernel(
    RasterParams P, const float4* __restrict__ packed, DirectSplats D,
    int32_t* __restrict__ pairs, int32_t* __restrict__ tile_starts,
    int32_t* __restrict__ tile_ends) {
  extern __shared__ uint16_t lds[];  // [kWaves][G] candidates
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tile = (int)blockIdx.x * kWaves + wave;
  if (tile >= P.num_tiles) return;  // (no barrier below)
  const int G = P.gpb;
  uint16_t* cand = lds + (int64_t)wave * G;
  const int img = tile / P.tiles_per_image;
  const int lt = tile - img * P.tiles_per_image;
  const uint32_t ty = (uint32_t)(lt / P.tiles_x);
  const uint32_t tx = (uint32_t)lt - ty * (uint32_t)P.tiles_x;
  const int64_t base = (int64_t)img * G;
  const uint64_t below = (1ull << lane) - 1ull;
  int n = 0;
  for (int g0 = 0; g0 < G; g0 += 64 * kBoxUnroll) {
    uint2 b[kBoxUnroll];
#pragma unroll
    for (int u = 0; u < kBoxUnroll; ++u)
      b[u] = D.box[base + min(g0 + 64 * u + lane, G - 1)];
#pragma unroll
    for (int u = 0; u < kBoxUnroll; ++u) {
      const int g = g0 + 64 * u + lane;
      const bool in = g < G && tx >= (b[u].x & 0xffffu) &&
                      tx <= (b[u].y & 0xffffu) && ty >= (b[u].x >> 16) &&
                      ty <= (b[u].y >> 16);
      const uint64_t m = __ballot(in);
      if (in) cand[n + __popcll(m & below)] = (uint16_t)g;
      n += __popcll(m);
    }
  }
  // (one wavefront: its LDS accesses take effect in program order)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float rx0, ry0, rx1, ry1;
  tile_rect((int)tx, (int)ty, P.width, P.height, rx0, ry0, rx1, ry1);
  const int start = tile * G;  // tiles x splats below 2^24: direct_ok
  int hits = 0;
  for (int c0 = 0; c0 < n; c0 += 64) {
    const bool ok = c0 + lane < n;
    const int64_t gid = base + cand[min(c0 + lane, n - 1)];
    const float4 p0 = packed[kRecordVec4 * gid];
    const float c = packed[kRecordVec4 * gid + 1].x;
    const float4 q = D.test[gid];
    const uint32_t f = __float_as_uint(q.w);
    ConicSlopes k;
    k.kc = q.y;
    k.ka = q.z;
    k.use_c = (f & 1u) != 0u;
    k.use_a = (f & 2u) != 0u;
    const bool hit = ok && ellipse_hits_rect(p0.x, p0.y, p0.z, p0.w, c, k, q.x,
                                             rx0, ry0, rx1, ry1);
    const uint64_t m = __ballot(hit);
    if (hit) pairs[start + hits + __popcll(m & below)] = (int32_t)gid;
    hits += __popcll(m);
  }
  if (lane == 0) {
    tile_starts[tile] = start;
    tile_ends[tile] = start + hits;
  }
}

}  // namespace

// Up to 4096 splats an image (LDS of the ranks; 64 box steps a tile) and
// 12.6M box tests in all (about 10 us of the chip): above, the five launches
// of the one-call binning cost less than the tests.
bool direct_ok(const RasterParams& P) {
  return P.num_tiles > 0 && P.num_splats > 0 && P.gpb <= kDirectMaxSplats &&
         P.tiles_x < (1 << 16) && P.tiles_y < (1 << 16) &&
         (int64_t)P.num_tiles * P.gpb <= kDirectMaxTests;
}

// The pairs that the compositors' workspace and variants go by: no count is
// taken here, and the lists' room (tiles x splats) is no measure of it.  Going
// by that room, images of more than a few tiles got a segment record per tile
// and, above 2048 tiles, the backward for long lists: 300 splats at 2048 x
// 2048 193 MB held for the backward and its kernel 18.7 us, now 134 and 15.5
// (by the pair count 102 and 14.7); 100 at 4096 x 4096 705 MB and 69, now 455
// and 57 (405, 57).  Long lists of faint splats lose nothing by the fewer
// records: 2000 large ones at 1080 x 1080 119 -> 117 us, 4096 at 850 x 850 329
// -> 246.
int64_t direct_pairs(const RasterParams& P) {
  return std::min((int64_t)P.num_tiles * P.gpb,
                  4 * (int64_t)P.num_tiles + (1 << 17));
}

int launch_direct_lists(const RasterParams& P, const float* means2d,
                        const float* conics, const float* colors,
                        const float* opacities, const float* depths,
                        float* packed, const DirectSplats& D, int32_t* pairs,
                        int32_t* tile_starts, int32_t* tile_ends,
                        const ZeroSpan zero[2], hipStream_t stream) {
  launch_traced(
      "direct_pack_kernel", direct_pack_kernel,
      dim3((unsigned)((P.gpb + kPackSplats - 1) / kPackSplats),
           (unsigned)P.batch),
      dim3(kPackThreads), 0, stream, P, means2d, conics, colors, opacities,
      depths, reinterpret_cast<float4*>(packed), D, zero[0], zero[1]);
  int rc = check_launch("direct_pack_kernel");
  if (rc) return rc;
  launch_traced("direct_list_kernel", direct_list_kernel,
                dim3((unsigned)((P.num_tiles + kWaves - 1) / kWaves)),
                dim3(kThreads), (size_t)kWaves * P.gpb * sizeof(uint16_t),
                stream, P, reinterpret_cast<const float4*>(packed), D, pairs,
                tile_starts, tile_ends);
  return check_launch("direct_list_kernel");
}

}  // namespace gs
