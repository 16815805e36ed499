// record.h -- the packed splat record, built by the binning (binning.hip) and
// the direct path (direct.hip).  Both are compiled with -ffp-contract=off and
// correctly rounded divisions and square roots.
#pragma once

#include "gs_internal.h"
#include "gs_predicate.h"
#define GS_HD __device__ __forceinline__
#include "gs_strip.h"

namespace gs {
namespace {

// Divisions and square roots of the per-splat strip constants: correctly
// rounded (this file is built with -fhip-fp32-correctly-rounded-divide-sqrt).
struct IeeeOps {
  static __device__ __forceinline__ float div(float x, float y) { return x / y; }
  static __device__ __forceinline__ float sqrt(float x) {
    return __builtin_sqrtf(x);
  }
};

// The packed 64-byte record of splat orig:
// {mx, my, a, b}, {c, o, r, g}, {b, slot | plain << 31, q, lo},
// {dxt, beta, gamma, delta}: lo = log2(o), q = plim + lo (the compositors'
// visibility bound on p + lo), plain = plain_record of the compositors'
// exponent coefficients, and the strip-culling constants (gs_strip.h).  The
// slot holds orig in the records of the compositors (pack_record) and the
// splat's tile-hit count in the original-order records of the count.
struct Record {
  float4 v[kRecordVec4];
};
__device__ __forceinline__ Record record_of(
    const RasterParams& P, const float* __restrict__ means2d,
    const float* __restrict__ conics, const float* __restrict__ colors,
    const float* __restrict__ opacities, int orig, uint32_t slot) {
  const float mx = means2d[2 * orig + 0];
  const float my = means2d[2 * orig + 1];
  const float a = conics[3 * orig + 0];
  const float b = conics[3 * orig + 1];
  const float c = conics[3 * orig + 2];
  const float o = opacities[orig];
  const float cr = colors[3 * orig + 0];
  const float cg = colors[3 * orig + 1];
  const float cb = colors[3 * orig + 2];
  const float plim = visibility_limit(o, P.alpha_thr, P.max_alpha);
  const float lo = opacity_log2(o);
  const bool plain = plain_record(
      (-0.5f * a) * kLog2e, (-b) * kLog2e, (-0.5f * c) * kLog2e, mx, my, o,
      plain_opacity_limit(fminf(P.max_alpha, 1.0f)));
  const StripConsts k = strip_consts_t<IeeeOps>(a, b, c, plim);
  Record r;
  r.v[0] = make_float4(mx, my, a, b);
  r.v[1] = make_float4(c, o, cr, cg);
  r.v[2] = make_float4(cb, __uint_as_float(slot | (plain ? 0x80000000u : 0u)),
                       plim + lo, lo);
  r.v[3] = make_float4(k.dxt, k.beta, k.gamma, k.delta);
  return r;
}

__device__ __forceinline__ void store_record(float4* __restrict__ dst,
                                             int64_t i, const Record& r) {
  float4* d = dst + (int64_t)kRecordVec4 * i;
#pragma unroll
  for (int k = 0; k < kRecordVec4; ++k) d[k] = r.v[k];
}

}  // namespace
}  // namespace gs
