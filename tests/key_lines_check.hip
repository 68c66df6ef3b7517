// The large-face pass's rows (gvv_raster.hpp BoxLines::start_rows) on projected triangles with boxes above
// 256 px, tall, wide and slivers: every pixel that the edge test passes must lie in its row's span
// (missed), and the 64-byte lines of visibility keys (8 keys of a row) that batches of 64 consecutive
// candidates touch are counted for tall boxes, with the lines that walking the box's longer side touches
// beside it.  Host only.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <utility>
#include "../gvv-differentiable-cuda-renderer_amd/csrc/gvv_raster.hpp"
using namespace gvv;

struct Counter {
  std::set<std::pair<int, int>> batch;
  int n = 0;
  long long lines = 0;
  void add(int x, int y) {
    batch.insert({y, x >> 3});
    if (++n == 64) done();
  }
  void done() {
    lines += (long long)batch.size();
    batch.clear();
    n = 0;
  }
};

static long long walk(const BoxLines& bl, int x0, int y0) {
  Counter c;
  for (int ln = 0; ln < bl.lines; ++ln) {
    int first;
    const int n = bl.span(ln, first);
    for (int k = first; k < first + n; ++k) c.add(x0 + (bl.columns ? ln : k), y0 + (bl.columns ? k : ln));
  }
  c.done();
  return c.lines;
}

int main(int argc, char** argv) {
  const int n = argc > 1 ? atoi(argv[1]) : 3000;
  std::mt19937 rng(9);
  std::uniform_real_distribution<float> U(0.f, 1.f);
  const int W = 1024, H = 1024;
  long long missed = 0, passed = 0, tall = 0, rows = 0, sides = 0;
  for (int t = 0; t < n; ++t) {
    const float sx = t % 3 == 0 ? 12.f + 30.f * U(rng) : 300.f * U(rng), sy = t % 3 == 1 ? 10.f : 60.f + 300.f * U(rng);
    const float cx = W * U(rng), cy = H * U(rng);
    float4 p[3];
    for (int k = 0; k < 3; ++k) p[k] = make_float4(cx + (U(rng) - 0.5f) * sx, cy + (U(rng) - 0.5f) * sy, 1000.f + 100.f * U(rng), 0.f);
    const Box bx = face_box(v3(p[0].x, p[0].y, p[0].z), v3(p[1].x, p[1].y, p[1].z), v3(p[2].x, p[2].y, p[2].z), W, H);
    if (bx.x0 > bx.x1 || bx.y0 > bx.y1) continue;
    const int bw = bx.x1 - bx.x0 + 1, bh = bx.y1 - bx.y0 + 1;
    if (bw * bh <= 256) continue;
    const EdgeTest et = edge_test(p[0], p[1], p[2]);
    BoxLines r, s;
    r.start_rows(et, bx.x0, bx.y0, bw, bh);
    s.start(et, bx.x0, bx.y0, bw, bh);
    if (r.columns || r.lines != bh || r.len != bw) { printf("not rows\n"); return 1; }
    for (int y = bx.y0; y <= bx.y1; ++y) {
      int first;
      const int cnt = r.span(y - bx.y0, first);
      for (int x = bx.x0; x <= bx.x1; ++x) {
        // the spans and the edge values round differently: a pixel that passes by less than the
        // rounding of either is the margin's to lose
        EdgeTest in = et;
        for (int k = 0; k < 3; ++k) in.c[k] -= 1e-3f;
        if (!in.pass(x + 0.5f, y + 0.5f)) continue;
        ++passed;
        missed += x - bx.x0 < first || x - bx.x0 >= first + cnt;
      }
    }
    if (bh > bw) {
      ++tall;
      rows += walk(r, bx.x0, bx.y0);
      sides += walk(s, bx.x0, bx.y0);
    }
  }
  printf("passed %lld missed %lld tall %lld row_lines %lld side_lines %lld\n", passed, missed, tall, rows, sides);
  return 0;
}
