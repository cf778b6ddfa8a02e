// raster_common.h -- what the rasterisers share: the staged form of a record,
// the coverage tests and one pixel's blend.
#pragma once
#include "spl_device.h"
#include "spl_internal.h"

namespace spl {

namespace {

// The fragment's Gaussian e^(-|tc|^2 / 2) (shaders.wgsl:586) is evaluated as
// 2^-(|S tc|^2) with S = sqrt(log2(e) / 2) folded into each entry's inverse
// map, so a pixel costs two fused products per coordinate and one exp2.
constexpr float kGaussScale = 0.84932180f;

// 2^y for y <= 0: y = k + f with k = rint(y), |f| <= 1/2, a degree-5
// relative minimax polynomial of 2^f (constant term 1, so exact at
// integers; within 3 ulp of exp2) in fused Horner form, then ldexp by k
// (exact while the result stays normal).  Only correctly rounded IEEE
// operations (fma, rint, ldexp), so it rounds the same on the CPU and the
// GPU.  The oracle clamps y at -125 first; below -8 every alpha is under the
// 1/255 fragment threshold either way, so the pixels agree without it.
__device__ __forceinline__ float spl_exp2(float y) {
  const float k = rintf(y);
  const float f = y - k;
  float p = 1.32764713e-3f;
  p = fmaf(p, f, 9.67554189e-3f);
  p = fmaf(p, f, 5.55071309e-2f);
  p = fmaf(p, f, 2.40221202e-1f);
  p = fmaf(p, f, 6.93146944e-1f);
  p = fmaf(p, f, 1.0f);
  return ldexpf(p, (int)k);
}

__device__ __forceinline__ float q8(float x) {
  x = fminf(fmaxf(x, 0.0f), 1.0f);
  return floorf(x * 255.0f + 0.5f);
}

__device__ __forceinline__ float clamp01(float x) { return fminf(fmaxf(x, 0.0f), 1.0f); }

// Pixel centres in the view plane are q = (sx px + ox, sy py + oy)
// (shaders.wgsl:561 inverted).  Each staged entry folds this map into its
// own: with e = o - t the coverage coordinate is affine in the integer
// pixel coordinates,
//   unaligned:     u = au px + bu py + cu,  w = av px + bv py + cv
//   axis-aligned:  dx = sx px + ex,  dy = sy py + ey  (then u, w from dx, dy)
// so a pixel costs two fused products per coordinate.
struct PixelMap {
  float sx, ox, sy, oy;
};

__device__ __forceinline__ PixelMap pixel_map(const Uniforms& u) {
  const float Wf = (float)u.image_size[0], Hf = (float)u.image_size[1], vw = u.view_size[0], vh = u.view_size[1];
  PixelMap p;
  p.sx = (2.0f * vw) / Wf;
  p.ox = vw / Wf - vw;
  p.sy = -(2.0f * vh) / Hf;
  p.oy = vh - vh / Hf;
  return p;
}

// The staged form of a record (g0: colour and opacity, g1: the rectangle's
// axes, g2: its centre and pixel box): e0 the inverse map scaled by S (and,
// unaligned, folded with the pixel map), e1 its translation, the coverage
// half-extent and the opacity, e2 the colour.
template <bool UNALIGNED>
__device__ __forceinline__ void prepare_entry(const float4& g0, const float4& g1, const float4& g2, const PixelMap& pm,
                                              float margin, float4& e0, float4& e1, float4& e2) {
  const float A00 = g1.x, A10 = g1.y, A01 = g1.z, A11 = g1.w;
  const float det = A00 * A11 - A10 * A01;
  const float rs = (1.0f / det) * kGaussScale;  // inverse map scaled by S
  const float i00 = A11 * rs, i01 = -A01 * rs, i10 = -A10 * rs, i11 = A00 * rs;
  const float ex = pm.ox - g2.x, ey = pm.oy - g2.y;
  // unaligned: the rectangle |tc| < margin in scaled coordinates;
  // axis-aligned: a square of half-side radius * margin in the view plane
  const float half = UNALIGNED ? margin * kGaussScale
                               : sqrtf(fmaxf(A00 * A00 + A10 * A10, A01 * A01 + A11 * A11)) * margin;
  if constexpr (UNALIGNED) {
    e0 = make_float4(i00 * pm.sx, i01 * pm.sy, i10 * pm.sx, i11 * pm.sy);
    e1 = make_float4(fmaf(i00, ex, i01 * ey), fmaf(i10, ex, i11 * ey), half, g0.w);
  } else {
    e0 = make_float4(i00, i01, i10, i11);
    e1 = make_float4(ex, ey, half, g0.w);
  }
  e2 = make_float4(g0.x, g0.y, g0.z, 0.0f);
}

// Can entry (m, t) cover a pixel centre of the pixel box [x0, x1] x
// [y0, y1]?  The tested coordinates are affine in the pixel, so their exact
// range over the box sits at the corners; the slack (relative to the
// magnitudes the per-pixel evaluation adds up) is far above its rounding.
template <bool UNALIGNED>
__device__ __forceinline__ bool range_meets(const float4& m, const float4& t, float x0, float x1, float y0, float y1,
                                            const PixelMap& pm) {
  const float h = t.z;
  float a0, a1, b0, b1, sa, sb;  // ranges of the tested coordinates, and slack
  if constexpr (UNALIGNED) {
    a0 = (fminf(m.x * x0, m.x * x1) + fminf(m.y * y0, m.y * y1)) + t.x;
    a1 = (fmaxf(m.x * x0, m.x * x1) + fmaxf(m.y * y0, m.y * y1)) + t.x;
    b0 = (fminf(m.z * x0, m.z * x1) + fminf(m.w * y0, m.w * y1)) + t.y;
    b1 = (fmaxf(m.z * x0, m.z * x1) + fmaxf(m.w * y0, m.w * y1)) + t.y;
    sa = 1e-4f * (((fabsf(m.x) * x1 + fabsf(m.y) * y1) + fabsf(t.x)) + h);
    sb = 1e-4f * (((fabsf(m.z) * x1 + fabsf(m.w) * y1) + fabsf(t.y)) + h);
  } else {
    a0 = fmaf(pm.sx, x0, t.x); a1 = fmaf(pm.sx, x1, t.x);  // sx > 0
    b0 = fmaf(pm.sy, y1, t.y); b1 = fmaf(pm.sy, y0, t.y);  // sy < 0
    sa = 1e-4f * ((pm.sx * x1 + fabsf(t.x)) + h);
    sb = 1e-4f * ((fabsf(pm.sy) * y1 + fabsf(t.y)) + h);
  }
  return a1 + sa >= -h && a0 - sa < h && b1 + sb >= -h && b0 - sb < h;
}

// Coverage of the pixel centre (pxf, pyf) by entry (m, t): the scaled
// texture coordinate (u, w2) and whether it lies in the rectangle.
template <bool UNALIGNED>
__device__ __forceinline__ bool covers(const float4& m, const float4& t, float pxf, float pyf, const PixelMap& pm,
                                       float& u, float& w2) {
  const float h = t.z;
  if constexpr (UNALIGNED) {
    u = fmaf(m.x, pxf, fmaf(m.y, pyf, t.x));  // S * texture coordinate
    w2 = fmaf(m.z, pxf, fmaf(m.w, pyf, t.y));
    return fmaxf(fabsf(u), fabsf(w2)) < h;
  } else {
    const float dx = fmaf(pm.sx, pxf, t.x), dy = fmaf(pm.sy, pyf, t.y);
    u = fmaf(m.x, dx, m.y * dy);
    w2 = fmaf(m.z, dx, m.w * dy);
    return fmaxf(fabsf(dx), fabsf(dy)) < h;
  }
}

// One pixel's blend state: colour and transmittance, unorm8 codes or f32.
template <bool F32>
struct PixelState {
  float c0 = 0.0f, c1 = 0.0f, c2 = 0.0f, tr = F32 ? 1.0f : 255.0f;

  // One fragment: alpha (shaders.wgsl:585-589) and the blend.  in: the
  // coverage test's verdict, for walks over candidates that did not pass
  // it yet; an uncovered fragment blends nothing.
  __device__ __forceinline__ void shade(float u, float w2, float opacity, const float4& col, bool in) {
    float alpha = opacity * spl_exp2(-fmaf(u, u, w2 * w2));
    if constexpr (!F32) {
      // unorm8 codes C, T: rint(s * T + C) (s clamped, sum capped at
      // 255) and rint(T * (1 - a)): the ideal 8-bit blender.  Below the
      // threshold alpha becomes 0, which leaves C and T as they are
      // (they hold integers; clamp01 of a NaN product is 0), so no
      // branch is needed.
      alpha = in && alpha >= 1.0f / 255.0f ? alpha : 0.0f;
      const float sr = col.x * alpha, sg = col.y * alpha, sb = col.z * alpha;
      // the source alpha needs no clamp: the opacity is a sigmoid (or 1
      // in the dev-test scene) and spl_exp2 of a non-positive argument is
      // at most 1 (p(f) <= p(0) = 1 when rint(y) = 0, p(f) / 2 < 1 below),
      // so alpha is in [0, 1] after the threshold
      const float sa = alpha;
      c0 = fminf(rintf(fmaf(clamp01(sr), tr, c0)), 255.0f);
      c1 = fminf(rintf(fmaf(clamp01(sg), tr, c1)), 255.0f);
      c2 = fminf(rintf(fmaf(clamp01(sb), tr, c2)), 255.0f);
      tr = rintf(fmaf(-sa, tr, tr));
    } else if (in && alpha >= 1.0f / 255.0f) {
      const float sr = col.x * alpha, sg = col.y * alpha, sb = col.z * alpha;
      const float da = tr;
      c0 = fmaf(sr, da, c0);
      c1 = fmaf(sg, da, c1);
      c2 = fmaf(sb, da, c2);
      tr = fmaf(-alpha, da, da);
    }
  }

  // The pixel's final value, as the frame stores it.
  __device__ __forceinline__ uint32_t packed(bool bgra) const {
    uint32_t r, g, b, al;
    if (!F32) {
      r = (uint32_t)c0; g = (uint32_t)c1; b = (uint32_t)c2; al = (uint32_t)tr;
    } else {
      r = (uint32_t)q8(c0); g = (uint32_t)q8(c1); b = (uint32_t)q8(c2); al = (uint32_t)q8(tr);
    }
    return bgra ? (b | (g << 8) | (r << 16) | (al << 24)) : (r | (g << 8) | (b << 16) | (al << 24));
  }
};

}  // namespace

}  // namespace spl
