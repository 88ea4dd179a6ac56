// Per-tile restaging of a raster record, shared by the plain and the
// differentiable rasters (device code).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"
#include "device.h"

namespace vkgs {

__device__ __forceinline__ uint32_t pack16(int lo, int hi) { return (uint32_t)lo | ((uint32_t)hi << 16); }

// A raster record (cx, cy, i00, i01), (i10, i11, opacity, x rect), (r, g, b,
// y rect) restaged for one tile (see kFrameScale): the scaled inverse
// rot_scale rows with their offsets at the corner (X0, Y0) of the tile's
// 64 x 64 pixel block, -log2(opacity), the colour and the pixel rectangle:
//   s0 = (i'00, i'01, o'x, -log2 opacity), s1 = (i'10, i'11, o'y, x rect),
//   s2 = (r, g, b, y rect).
// A lane with no record stages one that covers no pixel: offsets `inert`
// (+inf, or a large finite value where a zero weight multiplies the frame
// coordinates, which must stay finite) and an empty rectangle.
struct StagedRecord {
  float4 a, b, c;
};

__device__ __forceinline__ StagedRecord staged(const float4& p0, const float4& p1, const float4& p2, float X0,
                                               float Y0) {
  const float i00 = p0.z * kFrameScale, i01 = p0.w * kFrameScale;
  const float i10 = p1.x * kFrameScale, i11 = p1.y * kFrameScale;
  const float dx = X0 - p0.x, dy = Y0 - p0.y;
  return {make_float4(i00, i01, fmaf(i00, dx, i01 * dy), -__builtin_amdgcn_logf(p1.z)),
          make_float4(i10, i11, fmaf(i10, dx, i11 * dy), p1.w), p2};
}

__device__ __forceinline__ StagedRecord staged_inert(float inert) {
  const float empty = __uint_as_float(pack16(1, 0));
  return {make_float4(0.f, 0.f, inert, inert), make_float4(0.f, 0.f, inert, empty),
          make_float4(0.f, 0.f, 0.f, empty)};
}

__device__ __forceinline__ void stage_record(const float4& p0, const float4& p1, const float4& p2, bool valid,
                                             float X0, float Y0, float4* s0, float4* s1, float4* s2,
                                             float inert = __builtin_inff()) {
  const StagedRecord r = valid ? staged(p0, p1, p2, X0, Y0) : staged_inert(inert);
  *s0 = r.a;
  *s1 = r.b;
  *s2 = r.c;
}

// False only if the staged record covers no pixel of the 8x8 tile whose middle
// is (mx, my) from the block's corner: the tile lists hold every tile of a
// splat's rectangle, and of a slanted splat's the square misses many (17-36% of
// the pairs measured over cloud, street and city scenes).  Along each of the
// square's two axes the tile's pixel centres reach 3.5 (|x| + |y|) from the
// middle's coordinate.  `slack` is above the rounding of both sides (each two
// fused steps of terms below `size`); NaN and infinite rows keep the record.  A pixel
// that a kept record does not cover still adds its colour times 0: of an infinite or
// NaN colour that is NaN, so such a splat marks the tiles that it may cover, and no
// longer all of its rectangle's.
__device__ __forceinline__ bool axis_may_cover(const float4& r, float mx, float my) {
  const float step = fabsf(r.x) + fabsf(r.y);
  const float size = fmaf((float)kRasterBlock, step, fabsf(r.z));
  const float slack = fmaf(size, 0x1p-20f, 0x1p-16f);
  return !(fabsf(fmaf(r.x, mx, fmaf(r.y, my, r.z))) > fmaf(3.5f, step, kCoverScaled) + slack);
}
__device__ __forceinline__ bool may_cover8(const StagedRecord& r, float mx, float my) {
  return axis_may_cover(r.a, mx, my) & axis_may_cover(r.b, mx, my);
}

// Two 8x8 tiles per wave (lane l of half h):  where a lane's staged record goes in its tile's batch: the kept ones first, in
// lane order, the others after them; n_a and n_b records are kept of the two tiles.
struct PairSlots {
  uint64_t kept;  // bit 32 h + l: entry l of tile h's batch
  bool keep;
  int at, n_a, n_b;
};

__device__ __forceinline__ PairSlots pair_slots(bool keep, int h, int l) {
  const uint64_t m = __ballot(keep);
  PairSlots p;
  p.kept = m;
  p.keep = keep;
  p.n_a = __popc((uint32_t)m);
  p.n_b = __popc((uint32_t)(m >> 32));
  const int below = (int)mbcnt(m) - (h ? p.n_a : 0);
  p.at = keep ? below : (h ? p.n_b : p.n_a) + l - below;
  return p;
}

}  // namespace vkgs
