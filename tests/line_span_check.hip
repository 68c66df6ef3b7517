// The line spans of the depth pass (gvv_raster.hpp BoxLines) against the exact ray/triangle
// test: random triangles (a third slivers, some with a vertex far outside the image) seen by a
// pinhole camera, boxes clipped to the image, up to 4096 px and a few of any size.  Counts the pixels that the
// exact test accepts and the spans leave out (missed), and the least distance in px by which an
// accepted pixel lies inside an edge's bound (slack; the pre-test's margin is 1/32 px).
// Host only.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include "../gvv-differentiable-cuda-renderer_amd/csrc/gvv_raster.hpp"
using namespace gvv;
int main(int argc, char** argv) {
  const int ntri = argc > 1 ? atoi(argv[1]) : 20000;
  std::mt19937 rng(11);
  std::uniform_real_distribution<double> U(0, 1);
  std::normal_distribution<double> G(0, 1);
  long long accepted = 0, missed = 0, boxes = 0, kept = 0, area = 0;
  double slack = 1e9;
  for (int t = 0; t < ntri; ++t) {
    const int W = t % 5 == 0 ? 8192 : 1024, H = t % 7 == 0 ? 389 : 1024;
    // camera on the z axis looking at the origin, from 0.6 to 5 m
    const float dist = (float)(600.0 + 4400.0 * U(rng));
    const float E[12] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, dist};
    const float K[9] = {1.2f * W, 0, W / 2.f, 0, 1.2f * W, H / 2.f, 0, 0, 1};
    Camera cam;
    camera_setup(E, K, cam);
    const double px_mm = dist / (1.2 * W);
    const bool big = t % 997 == 0;
    const double size = px_mm * std::pow(10.0, -0.5 + 2.2 * U(rng)) * (big ? 30 : 1);      // 0.3 .. 50 px
    const double cx = (U(rng) - 0.5) * W * px_mm, cy = (U(rng) - 0.5) * H * px_mm, cz = G(rng) * 50;
    V3 v[3];
    float4 p[3];
    for (int k = 0; k < 3; ++k) {
      const double s2 = t % 3 == 2 ? 0.02 : 1.0, far = t % 11 == 0 && k == 2 ? 40.0 : 1.0;
      const double a = G(rng) * size * far, b = G(rng) * size * (k == 1 ? s2 : 1.0);
      v[k] = t % 2 ? v3((float)(cx + a), (float)(cy + b), (float)(cz + G(rng) * size))
                   : v3((float)(cx + b), (float)(cy + a), (float)(cz + G(rng) * size));
      if (t % 13 == 0 && k == 1) v[k].y = v[0].y;                          // an edge parallel to the rows
      const V3 q = project(cam, v[k]);
      p[k] = make_float4(q.x, q.y, q.z, 0.f);
    }
    const Box bx = face_box(v3(p[0].x, p[0].y, p[0].z), v3(p[1].x, p[1].y, p[1].z), v3(p[2].x, p[2].y, p[2].z), W, H);
    if (bx.x0 > bx.x1 || bx.y0 > bx.y1) continue;
    const int bw = bx.x1 - bx.x0 + 1, bh = bx.y1 - bx.y0 + 1;
    if ((long long)bw * bh > 4096 && !big) continue;
    ++boxes;
    area += bw * bh;
    const EdgeTest et = edge_test(p[0], p[1], p[2]);
    const TriSetup ts = tri_setup(v[0], v[1], v[2]);
    BoxLines bl;
    bl.start(et, bx.x0, bx.y0, bw, bh);
    for (int ln = 0; ln < bl.lines; ++ln) {
      int first;
      const int n = bl.span(ln, first);
      kept += n;
      if (n < 0 || (n > 0 && (first < 0 || first + n > bl.len))) { printf("bad span\n"); return 1; }
      for (int k = 0; k < bl.len; ++k) {
        const int x = bx.x0 + (bl.columns ? ln : k), y = bx.y0 + (bl.columns ? k : ln);
        const V3 abc = ray_barycentric(ts, cam_origin_scaled(cam), pixel_ray(cam, x + 0.5f, y + 0.5f));
        if (!inside(abc)) continue;
        ++accepted;
        if (k < first || k >= first + n) ++missed;
        for (int i = 0; i < 3; ++i) {
          const double ea = bl.columns ? et.b[i] : et.a[i];
          const double b = (double)bl.t[i] + (double)ln * bl.s[i];
          const double d = bl.lower[i] ? (k - b) * ea : bl.upper[i] ? (k - b) * ea : 1e9;
          if (d < slack) slack = d;
        }
      }
    }
  }
  printf("boxes %lld area %lld kept %lld accepted %lld missed %lld slack %.6e margin %.6e\n", boxes, area, kept, accepted,
         missed, slack, (double)kEdgeMargin);
  return 0;
}
