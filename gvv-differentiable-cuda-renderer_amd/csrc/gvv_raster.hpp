// gvv_raster.hpp -- screen-space pre-test of the depth pass: the conservative edge test and
// the per-row spans it implies.  Host- and device-callable so that its conservativeness can be
// checked on the CPU.
#pragma once
#include "gvv_math.hpp"

namespace gvv {

// Conservative screen-space pre-test.  A pixel passes the exact ray/triangle test only if its
// centre lies inside the projected triangle up to the float error of that test (ray/triangle
// barycentrics below zero are rejected outright), so every pixel farther than kEdgeMargin px
// outside an edge can be skipped without changing any result.  Over 2e8 pixel tests of random
// triangles at the renderer's scale the farthest accepted pixel lay 7e-4 px outside an edge
// (tests/edge_margin_check.hip), so 1/32 px leaves a factor of 45.  The pre-test is disabled
// (every bounding-box pixel takes the exact test) when a vertex is near or behind the camera
// plane, when coordinates are huge (beyond 65536 px an edge value's own rounding, 3 ulp of the
// coordinate, would come near the margin), or when the projected triangle is degenerate.
constexpr float kEdgeMargin = 0.03125f;

struct EdgeTest {
  float a[3], b[3], c[3];
  bool on;
  GVV_HD bool pass(float x, float y) const {
    if (!on) return true;
    return (a[0] * x + b[0] * y + c[0] >= 0.f) && (a[1] * x + b[1] * y + c[1] >= 0.f) &&
           (a[2] * x + b[2] * y + c[2] >= 0.f);
  }
};

GVV_HD EdgeTest edge_test(float4 p0, float4 p1, float4 p2) {
  EdgeTest e;
  e.on = false;
  const float px[3] = {p0.x, p1.x, p2.x}, py[3] = {p0.y, p1.y, p2.y}, pz[3] = {p0.z, p1.z, p2.z};
  for (int i = 0; i < 3; ++i)
    if (!(pz[i] >= 1.0f) || !(fabsf(px[i]) <= 65536.f) || !(fabsf(py[i]) <= 65536.f)) return e;
  const float area2 = (px[1] - px[0]) * (py[2] - py[0]) - (py[1] - py[0]) * (px[2] - px[0]);
  if (!(fabsf(area2) >= 1e-3f)) return e;
  const float s = area2 > 0.f ? 1.f : -1.f;
  for (int i = 0; i < 3; ++i) {
    const int j = (i + 1) % 3;
    const float ex = px[j] - px[i], ey = py[j] - py[i];
    const float len = sqrtf(ex * ex + ey * ey);
    if (!(len > 0.f)) return e;
    // signed distance of (x, y) to edge i, positive inside: s * cross(e, p - p_i) / |e|
    e.a[i] = -s * ey / len;
    e.b[i] = s * ex / len;
    e.c[i] = -(e.a[i] * px[i] + e.b[i] * py[i]) + kEdgeMargin;
  }
  e.on = true;
  return e;
}

// The pre-test walked along the rows of a box: the three edge values at the current pixel are
// kept and advanced by a (one pixel along a row) or, at a row end, by b - (bw - 1) a (back to
// the row's first pixel, one row down), instead of being evaluated anew at every pixel.  The
// stepped values differ from the direct ones by rounding only (at most 64 steps of values
// under 100 px), far inside the margin; tests/edge_margin_check.hip runs this walk over every
// box it draws and counts the accepted pixels that it would reject (none).
struct EdgeWalk {
  float e[3];     // edge values at the current pixel
  float w[3];     // row-end step b - (bw - 1) a
  GVV_HD void start(const EdgeTest& t, int x0, int y0, int bw) {
    const float x = x0 + 0.5f, y = y0 + 0.5f;
    for (int i = 0; i < 3; ++i) {
      e[i] = t.a[i] * x + t.b[i] * y + t.c[i];
      w[i] = t.b[i] - (float)(bw - 1) * t.a[i];
    }
  }
  GVV_HD bool pass(bool on) const { return !on || (e[0] >= 0.f && e[1] >= 0.f && e[2] >= 0.f); }
  GVV_HD void step(const EdgeTest& t, bool row_end) {
    for (int i = 0; i < 3; ++i) e[i] += row_end ? w[i] : t.a[i];
  }
};

// Approximate reciprocal and reciprocal square root (1 ulp on the device): only for the
// pre-test, whose margin is thousands of times their rounding.
GVV_HD float approx_rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.f / x;
#endif
}

// The pixels of a box that the pre-test keeps, line by line: lines run along the box's longer
// side (rows, or columns of a tall box), and on each line the kept pixels are one interval,
// because each edge bounds the position along the line from one side.  An edge's bound moves
// linearly from line to line (t + ln * s), so a line costs three FMAs instead of three edge
// values per pixel.
// Rounding: with e0 the edge value at the box's first pixel and ea the edge's slope along the
// line, a bound is -(e0 + el ln) / ea.  Its error is a few ulp of the edge value's terms (under
// 2e-3 px for coordinates up to 65536, the limit of edge_test) divided by |ea|, while the
// margin moves the bound outwards by kEdgeMargin / |ea|: the margin's factor over the error
// does not depend on ea.  An edge parallel to the lines (ea = 0) bounds nothing here.
struct BoxLines {
  float t[3], s[3];            // bound of edge i on line ln, in pixels from the line's start
  bool lower[3], upper[3];     // which side it bounds
  int lines, len;              // lines of the box and pixels per line
  bool columns;                // lines are columns (the box is taller than wide)
  GVV_HD void start(const EdgeTest& e, int x0, int y0, int bw, int bh) {
    columns = bh > bw;
    lines = columns ? bw : bh;
    len = columns ? bh : bw;
    const float x = x0 + 0.5f, y = y0 + 0.5f;
    for (int i = 0; i < 3; ++i) {
      const float ea = columns ? e.b[i] : e.a[i], el = columns ? e.a[i] : e.b[i];
      const float r = approx_rcp(ea);
      t[i] = -(e.a[i] * x + e.b[i] * y + e.c[i]) * r;
      s[i] = -el * r;
      lower[i] = e.on && ea > 0.f;
      upper[i] = e.on && ea < 0.f;
    }
  }
  // first kept pixel of line ln and how many follow from it (0: none); NaN bounds (an infinite
  // slope at line 0) bound nothing
  GVV_HD int span(int ln, int& first) const {
    float lo = 0.f, hi = (float)(len - 1);
    for (int i = 0; i < 3; ++i) {
      const float b = fmaf((float)ln, s[i], t[i]);
      if (lower[i]) lo = fmaxf(lo, b);
      if (upper[i]) hi = fminf(hi, b);
    }
    first = 0;
    if (!(lo <= hi)) return 0;
    first = (int)ceilf(lo);
    return (int)floorf(hi) - first + 1;
  }
};

// Conservative x-range [xl, xr] of bounding-box row y (pixel centres at y + 0.5) inside the
// three half-planes of the edge pre-test, widened by one pixel on each side so that float
// rounding of the bounds never drops a pixel the pre-test would pass.  Without a usable edge
// test the whole row is returned.
GVV_HD void row_span(const EdgeTest& e, int y, int x0, int x1, int& xl, int& xr) {
  xl = x0;
  xr = x1;
  if (!e.on) return;
  const float yc = y + 0.5f;
  float lo = (float)x0, hi = (float)x1;    // range of pixel indices x (centre x + 0.5)
  for (int i = 0; i < 3; ++i) {
    const float rhs = -(e.b[i] * yc + e.c[i]);      // need a * xc >= rhs
    if (e.a[i] > 0.f) lo = fmaxf(lo, rhs / e.a[i] - 1.5f);
    else if (e.a[i] < 0.f) hi = fminf(hi, rhs / e.a[i] + 0.5f);
    else if (rhs > 1.f) hi = lo - 1.f;              // horizontal edge with the row well outside
  }
  if (!(lo <= hi)) { xr = x0 - 1; return; }         // empty (also catches NaN)
  xl = (int)floorf(lo);
  xr = (int)ceilf(hi);
  if (xl < x0) xl = x0;
  if (xr > x1) xr = x1;
}

}  // namespace gvv
