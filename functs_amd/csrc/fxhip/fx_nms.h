// What the kernels of the detection tail share (fx_nms.hip, fx_nms_pairs.hip): the order of the keys
// and the overlap test.
#pragma once
#include "fx_device.h"

namespace {

__device__ __forceinline__ uint32_t orderable(float f) {   // monotone map float -> uint32
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float from_orderable(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}

struct Box { float x1, y1, x2, y2; };

__device__ __forceinline__ bool overlaps(const Box& a, float area_a, const Box& b, float area_b, float thr) {
  const float xx1 = fmaxf(a.x1, b.x1), yy1 = fmaxf(a.y1, b.y1);
  const float xx2 = fminf(a.x2, b.x2), yy2 = fminf(a.y2, b.y2);
  const float w = fmaxf(0.0f, xx2 - xx1), h = fmaxf(0.0f, yy2 - yy1);
  const float inter = w * h;
  const float iou = inter / ((area_a + area_b) - inter);
  return iou > thr;
}

// The same decision without the division, where that is certain: inter / union > thr is settled by
// comparing inter with thr * union unless the two are within 2e-6 of each other (the product and the
// quotient are off by at most 2^-24 relative each, 2e-6 is 2^-19), or the product is not an ordinary
// number (boxes of no or infinite area, NaN) or thr is not positive (boxes with swapped corners may make the
// union negative, and dividing by it turns the comparison round: with thr < 0 the product would be an
// ordinary number all the same).
__device__ __forceinline__ void overlaps_fast(const Box& a, float area_a, const Box& b, float area_b, float thr, bool& over, bool& sure) {
  const float xx1 = fmaxf(a.x1, b.x1), yy1 = fmaxf(a.y1, b.y1);
  const float xx2 = fminf(a.x2, b.x2), yy2 = fminf(a.y2, b.y2);
  const float w = fmaxf(0.0f, xx2 - xx1), h = fmaxf(0.0f, yy2 - yy1);
  const float inter = w * h;
  const float t = thr * ((area_a + area_b) - inter);
  over = inter > t * 1.000002f;
  sure = thr > 0.0f && t > 1e-30f && t < 1e30f && (over || inter < t * 0.999998f);
}

// The lanes of the wave in which the two may overlap: boxes apart from each other are told by four comparisons (no overlap
// passes a positive threshold, whatever the areas), and most waves hold no others.  Masks, not a branch a lane: what the
// compiler makes of the latter is four times the instructions.
__device__ __forceinline__ uint64_t near_lanes(const float4& a, const float4& b, float thr) {
  const uint64_t near = __ballot(a.z > b.x) & __ballot(b.z > a.x) & __ballot(a.w > b.y) & __ballot(b.w > a.y);
  return thr > 0.0f ? near : ~0ull;
}
// of those lanes the ones in which they do: the decisions of overlaps(), by the division for waves in which a lane needs it
__device__ __forceinline__ uint64_t overlap_lanes(uint64_t near, const float4& a, float area_a, const float4& b, float area_b, float thr) {
  const Box p{a.x, a.y, a.z, a.w}, q{b.x, b.y, b.z, b.w};
  bool over, sure;
  overlaps_fast(p, area_a, q, area_b, thr, over, sure);
  uint64_t lanes = __ballot(over);
  const uint64_t open = __ballot(!sure) & near;
  if (open != 0ull) lanes = (lanes & ~open) | (__ballot(overlaps(p, area_a, q, area_b, thr)) & open);
  return lanes & near;
}

}  // namespace
