// gvv_raster.hpp -- screen-space pre-test of the depth pass: the conservative edge test and
// the per-row spans it implies.  Host- and device-callable so that its conservativeness can be
// checked on the CPU.
#pragma once
#include "gvv_math.hpp"

namespace gvv {

// Conservative screen-space pre-test.  A pixel passes the exact ray/triangle test only if its
// centre lies inside the projected triangle up to the binary32 errors of that test and of the
// projection (ray/triangle barycentrics below zero are rejected outright), so every pixel farther
// than that outside an edge can be skipped without changing any result.  The margin of a face is
// at least kEdgeMargin, and a bound of those errors where that is larger: over 2e8 pixel tests of
// random triangles at the renderer's scale the farthest accepted pixel lay 7e-4 px outside an edge
// (tests/edge_margin_check.hip), but a needle 1 mm wide and 1 m long is accepted up to half a pixel
// outside, and a face that reaches a few mm from the camera several pixels.
//
// The bound, with u = 2^-24.  Exact is the projection of the binary32 vertices by the binary32 E and
// K; P is the test's hit point, accepted by its three half-planes.
//   normal       N = e1 x e2 in binary32 is tilted against the plane by up to 7 u q, q = L^2 / |N|
//                (L: longest edge; q is 2 for an equilateral triangle, 1000 for the needle).  The
//                half-planes contain their edges but run along N, so over a distance L a point of
//                the plane lies up to 9 u q L beside the hit point
//   hit point    dot(v0, N) - dot(o, N), dot(d, N), their quotient and o + t d: 12 u (|V| + |o|) off
//                the plane; the ray's normalised direction, the origin's and the vertices' scaling
//                by 1/1000: 9 u (|V| + |o|) beside the ray
//   half-planes  N . (e x (P - v)) in binary32: 18 u L beside an edge
// all three in world units, times gs / z in pixels: gs bounds the derivative of the projection over
// the image (view_error), z is the least depth of the vertices.  In pixels:
//   ray          the binary32 inverse of K E and the ray origin against E and K: their residuals, formed
//                in binary64 per view, and the rounding of the back-projected point
//   projection   7 u (|K| (|E| |V| + |t|)) / z per vertex; a point of the triangle moves by no more
//                than its vertices, so an edge does too
//   edge values  coefficients and evaluation: 38 u times the largest coordinate
// All but the last are sums over the vertices weighted by the point's barycentrics in the image, so
// their maximum bounds them; where that is above kEdgeMargin, the weights are bounded over the box
// (a vertex far off screen, whose own error may be hundreds of px, moves the edges on the screen by
// a small share of it: 4,000 faces that each reach to 1.5-20 mm from the camera, 4 views of 512^2,
// forward 8.8 ms by the maximum alone, 5.5 ms so, 7.1 with the fixed margin, which loses pixels).
// A projected triangle thinner than its vertices' errors (seen edge-on) can turn its edges by any
// angle; there a point within the half-planes has barycentrics above -10 u q, in the image up to
// zr = zmax / zmin times as much, of a height of at most its longest edge.
// The pre-test is disabled (every bounding-box pixel takes the exact test) when a vertex is near
// or behind the camera plane, coordinates are beyond 1e6 px, the projected triangle is degenerate (the
// sign of its area uncertain), or q zr > 1e5, from where the bound's own terms no longer hold.
// Each bound is an upper one of sums that mostly cancel; tests/pretest_cover_check.hip draws the
// cases above and finds accepted pixels out to 0.22 of a face's margin (with kEdgeMargin alone, up to
// one accepted pixel in 260 is lost there).  At 1024 px, f = 1229 px and cameras 3 to 3.5 m away the
// bound of an ordinary face is 0.018 px, so its margin is kEdgeMargin.  The terms take the setup and
// vertex launches 1.5 us of 25 (100k faces over 8 x 1024^2), the depth passes nothing measurable.
constexpr float kEdgeMargin = 0.03125f;
constexpr float kUnit = 0x1p-24f;

// Approximate reciprocal and reciprocal square root (1 ulp on the device): only for the
// pre-test, whose margin is thousands of times their rounding.
GVV_HD float approx_rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.f / x;
#endif
}

// Two positive floats as the halves of a word, 8 significant bits each, rounded up; anything that is
// not a number below 2^100 becomes infinity.  Words compare as their first floats.
GVV_HD uint32_t half_up(float x) {
  if (!(x < 0x1p100f)) return 0x7f80u;
  uint32_t b;
  __builtin_memcpy(&b, &x, 4);
  return (b + 0xffffu) >> 16;
}
GVV_HD uint32_t pack_up(float hi, float lo) { return (half_up(hi) << 16) | half_up(lo); }
GVV_HD float float_of(uint32_t b) {
  float x;
  __builtin_memcpy(&x, &b, 4);
  return x;
}
GVV_HD float hi_float(uint32_t w) { return float_of(w & 0xffff0000u); }
GVV_HD float lo_float(uint32_t w) { return float_of(w << 16); }

// The terms of a view (one thread of the setup launch each): the error in px of a vertex V at
// depth z that projects to p is c + (cz + cv |V| + |p| (pz + pv |V|)) / z, and a world-space error
// of 1 at depth z is at most gs / z px.
struct ViewError {
  float c, cz, cv, pz, pv, gs;
};

GVV_HD ViewError view_error(const Camera& cam, int W, int H) {
  // M = K E and what K E (K E)^-1 leaves of the back-projected homogeneous pixel (x z, y z, z, 1)
  const double h[4] = {1000.0 * W, 1000.0 * H, 1000.0, 1.0};
  float m[3][3], dev[3], org[3], kE[3], kT[3], sT = 0.f;
  for (int r = 0; r < 3; ++r) {
    double mr[4];
    for (int k = 0; k < 4; ++k) {
      mr[k] = 0.0;
      for (int j = 0; j < 3; ++j) mr[k] += (double)cam.K[3 * r + j] * (double)cam.E[4 * j + k];
    }
    double d = 0.0, o = mr[3];
    for (int k = 0; k < 4; ++k) {
      double t = (k == 3 ? mr[3] : 0.0) - (k == r ? 1.0 : 0.0);
      for (int j = 0; j < 3; ++j) t += mr[j] * (double)cam.invP[4 * j + k];
      d += fabs(t) * h[k];
    }
    for (int j = 0; j < 3; ++j) o += mr[j] * (double)cam.o[j];
    dev[r] = (float)d;
    org[r] = fabsf((float)o);
    float s = 0.f;
    kE[r] = kT[r] = 0.f;
    for (int j = 0; j < 3; ++j) {
      m[r][j] = (float)mr[j];
      const float k = fabsf(cam.K[3 * r + j]);
      const float* e = cam.E + 4 * j;
      kE[r] += k * fmaxf(fabsf(e[0]), fmaxf(fabsf(e[1]), fabsf(e[2])));
      kT[r] += k * fabsf(e[3]);
    }
    for (int k = 0; k < 4; ++k) s += fabsf(cam.invP[4 * r + k]) * (float)h[k];
    sT = fmaxf(sT, s);
  }
  const float wx = (float)W, wy = (float)H;
  float g[2] = {0.f, 0.f};             // |m0 - x m2|^2 and |m1 - y m2|^2 at the far ends of the image
  for (int c = 0; c < 2; ++c)
    for (int end = 0; end < 2; ++end) {
      const float x = end ? (c ? wy : wx) : 0.f;
      float q = 0.f;
      for (int j = 0; j < 3; ++j) q += (m[c][j] - x * m[2][j]) * (m[c][j] - x * m[2][j]);
      g[c] = fmaxf(g[c], q);
    }
  ViewError v;
  v.gs = 1.01f * sqrtf(g[0] + g[1]);
  const float ray = dev[0] + dev[1] + (wx + wy) * dev[2], org_px = org[0] + org[1] + (wx + wy) * org[2];
  const float o1 = fabsf(cam.o[0]) + fabsf(cam.o[1]) + fabsf(cam.o[2]);
  v.c = 1.2e-3f * (ray + org_px) + kUnit * (9.f * 1e-3f * sT * v.gs + 38.f * fmaxf(wx, wy));
  v.cz = 1.6f * org_px + kUnit * (32.f * o1 * v.gs + 12.f * (kT[0] + kT[1]));
  v.cv = kUnit * (32.f * v.gs + 12.f * (kE[0] + kE[1]));
  v.pz = kUnit * 12.f * kT[2];
  v.pv = kUnit * 12.f * kE[2];
  if (!(dev[2] < 100.f)) v.c = 0x1p120f;           // the inverse is none: no pre-test
  return v;
}

// The margin terms of a vertex, kept beside its projection: its error in px and gs / z.
GVV_HD float vertex_error(const ViewError& e, V3 v, V3 p) {
  const float v1 = fabsf(v.x) + fabsf(v.y) + fabsf(v.z), px = fmaxf(fabsf(p.x), fabsf(p.y));
  const float r = approx_rcp(p.z), dz = e.pz + e.pv * v1;
  float err = e.c + (e.cz + e.cv * v1 + px * dz) * r + 3.f * kUnit * px;
  if (!(dz * r <= 0.125f)) err = 0x1p120f;          // the depth itself is uncertain
  return float_of(pack_up(err, e.gs * r));
}

// The margin terms of a face's shape: the world-space errors in px per gs / z, and q.
GVV_HD uint32_t face_shape(const TriSetup& t) {
  const V3 a = t.v1 - t.v0, b = t.v2 - t.v1, c = t.v0 - t.v2;
  const float l2 = fmaxf(dot(a, a), fmaxf(dot(b, b), dot(c, c))), n2 = dot(t.N, t.N);
  if (!(n2 > 1e-30f)) return pack_up(0x1p120f, 0x1p120f);
  const float q = 1.01f * l2 * approx_rcp(sqrtf(n2));
  return pack_up(kUnit * 1330.f * sqrtf(l2) * (9.f * q + 66.f), q);
}

struct EdgeTest {
  float a[3], b[3], c[3];
  bool on;
  GVV_HD bool pass(float x, float y) const {
    if (!on) return true;
    return (a[0] * x + b[0] * y + c[0] >= 0.f) && (a[1] * x + b[1] * y + c[1] >= 0.f) &&
           (a[2] * x + b[2] * y + c[2] >= 0.f);
  }
};

// p: projected vertices with vertex_error in w (0: no error); shape: face_shape of the face; box: the
// pixels in question.
GVV_HD EdgeTest edge_test(float4 p0, float4 p1, float4 p2, uint32_t shape, const Box& box) {
  EdgeTest e;
  e.on = false;
  const float px[3] = {p0.x, p1.x, p2.x}, py[3] = {p0.y, p1.y, p2.y}, pz[3] = {p0.z, p1.z, p2.z};
  float pm = 0.f;
  for (int i = 0; i < 3; ++i) {
    if (!(pz[i] >= 1.0f) || !(fabsf(px[i]) <= 1e6f) || !(fabsf(py[i]) <= 1e6f)) return e;
    pm = fmaxf(pm, fmaxf(fabsf(px[i]), fabsf(py[i])));
  }
  const float area2 = (px[1] - px[0]) * (py[2] - py[0]) - (py[1] - py[0]) * (px[2] - px[0]);
  if (!(fabsf(area2) >= 1e-3f)) return e;
  float ex[3], ey[3], len[3], longest = 0.f;
  for (int i = 0; i < 3; ++i) {
    const int j = (i + 1) % 3;
    ex[i] = px[j] - px[i];
    ey[i] = py[j] - py[i];
    len[i] = sqrtf(ex[i] * ex[i] + ey[i] * ey[i]);
    if (!(len[i] > 0.f)) return e;
    longest = fmaxf(longest, len[i]);
  }
  const float area_unit = kUnit * longest * longest;      // 8 of these bound the area's rounding
  if (!(fabsf(area2) >= 12.f * area_unit)) return e;
  const float s = area2 > 0.f ? 1.f : -1.f;
  for (int i = 0; i < 3; ++i) {
    // signed distance of (x, y) to edge i, positive inside: s * cross(e, p - p_i) / |e|
    e.a[i] = -s * ey[i] / len[i];
    e.b[i] = s * ex[i] / len[i];
    e.c[i] = -(e.a[i] * px[i] + e.b[i] * py[i]);
  }
  // the margin: what each vertex adds, the largest of them, and the sum of each times the edge opposite
  const float w[3] = {p0.w, p1.w, p2.w};
  float err[3], most = 0.f, turn = 0.f;
  for (int i = 0; i < 3; ++i) {
    uint32_t b;
    __builtin_memcpy(&b, &w[i], 4);
    err[i] = hi_float(b) + hi_float(shape) * lo_float(b);
    most = fmaxf(most, err[i]);
    turn += err[i] * len[(i + 1) % 3];
  }
  const float rz = approx_rcp(fminf(pz[0], fminf(pz[1], pz[2])));
  const float q = lo_float(shape), qz = q * fmaxf(pz[0], fmaxf(pz[1], pz[2])) * rz;
  const float edges = 38.f * kUnit * pm;
  float bound = most + edges;
  if (!(turn + 100.f * area_unit <= 0.125f * fabsf(area2))) {
    bound += 14.f * kUnit * qz * longest;
  } else if (bound > kEdgeMargin) {
    // a vertex's error counts by its barycentric over the box
    const float x[2] = {box.x0 + 0.5f, box.x1 + 0.5f}, y[2] = {box.y0 + 0.5f, box.y1 + 0.5f};
    const float ra = approx_rcp(fabsf(area2));
    float sum = 0.f;
    for (int i = 0; i < 3; ++i) {
      const int j = (i + 1) % 3;           // the edge opposite
      const float d = e.c[j] + fmaxf(e.a[j] * x[0], e.a[j] * x[1]) + fmaxf(e.b[j] * y[0], e.b[j] * y[1]);
      sum += err[i] * (fminf(fmaxf(d, 0.f) * len[j] * ra, 1.25f) + 11.f * kUnit * q * pz[i] * rz);
    }
    bound = fminf(bound, 1.4f * sum + 1.25f * edges);
  }
  if (!(qz <= 1e5f) || !(bound <= 1e5f)) return e;
  const float margin = fmaxf(kEdgeMargin, bound);
  for (int i = 0; i < 3; ++i) e.c[i] += margin;
  e.on = true;
  return e;
}

// The same of a face without errors of its own (kEdgeMargin alone).
GVV_HD EdgeTest edge_test(float4 p0, float4 p1, float4 p2) { return edge_test(p0, p1, p2, 0u, Box{0, 0, 0, 0}); }

// The pre-test walked along the rows of a box: the three edge values at the current pixel are
// kept and advanced by a (one pixel along a row) or, at a row end, by b - (bw - 1) a (back to
// the row's first pixel, one row down), instead of being evaluated anew at every pixel.  The
// stepped values differ from the direct ones by rounding only (at most 64 steps of values
// under 100 px), far inside the margin; tests/edge_margin_check.hip runs this walk over every
// box it draws and counts the accepted pixels that it would reject (none).  The depth pass has
// walked lines (BoxLines) since; only that check uses this walk.
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

// The pixels of a box that the pre-test keeps, line by line: lines run along the box's longer
// side (rows, or columns of a tall box: start) or along its rows (start_rows), and on each line the kept pixels are one interval,
// because each edge bounds the position along the line from one side.  An edge's bound moves
// linearly from line to line (t + ln * s), so a line costs three FMAs instead of three edge
// values per pixel.
// Rounding: with e0 the edge value at the box's first pixel and ea the edge's slope along the
// line, a bound is -(e0 + el ln) / ea.  Its error is a few ulp of the edge value's terms (part of
// edge_test's 38 u times the largest coordinate) divided by |ea|, and the margin moves the bound
// outwards by margin / |ea|, so that one exceeds the other whatever ea is.  An edge parallel to the
// lines (|ea| below kLineSlope, from where 1 / ea times a coordinate stays finite) bounds nothing here.
constexpr float kLineSlope = 0x1p-60f;
struct BoxLines {
  float t[3], s[3];            // bound of edge i on line ln, in pixels from the line's start
  bool lower[3], upper[3];     // which side it bounds
  int lines, len;              // lines of the box and pixels per line
  bool columns;                // lines are columns (the box is taller than wide)
  GVV_HD void start(const EdgeTest& e, int x0, int y0, int bw, int bh) { start_lines(e, x0, y0, bw, bh, bh > bw); }
  // rows of any box, for faces of many pixels: along a row 8 visibility keys share a 64-byte line of
  // memory, along a column each has its own
  GVV_HD void start_rows(const EdgeTest& e, int x0, int y0, int bw, int bh) { start_lines(e, x0, y0, bw, bh, false); }
  GVV_HD void start_lines(const EdgeTest& e, int x0, int y0, int bw, int bh, bool by_columns) {
    columns = by_columns;
    lines = columns ? bw : bh;
    len = columns ? bh : bw;
    const float x = x0 + 0.5f, y = y0 + 0.5f;
    for (int i = 0; i < 3; ++i) {
      const float ea = columns ? e.b[i] : e.a[i], el = columns ? e.a[i] : e.b[i];
      const float r = approx_rcp(ea);
      t[i] = -(e.a[i] * x + e.b[i] * y + e.c[i]) * r;
      s[i] = -el * r;
      lower[i] = e.on && ea > kLineSlope;
      upper[i] = e.on && ea < -kLineSlope;
    }
  }
  // first kept pixel of line ln and how many follow from it (0: none)
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
// test the whole row is returned.  The kernels take BoxLines' spans; tests/raster_span_check.hip
// alone uses this.
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
