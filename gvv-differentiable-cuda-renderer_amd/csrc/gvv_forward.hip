// gvv_forward.hip -- forward kernels of the rasterizer (gfx950).
//
// Replaces renderBuffersGPU (reference cpp/src/Renderer/CUDABasedRasterization.cu:449-473):
//   k_setup         one launch for the short stages: per-view inverse matrices and ray origin
//                   (.cu:23-67); unnormalised world-space face normals and the scaled
//                   ray/triangle constants, once per mesh and face rather than per view
//                   (.cu:122-141); zero fills (the backward's gradient buffers)
//   k_vertices      vertex normals by CSR gather + per-view projection  (.cu:98-115,148-174)
//   k_raster        per (view, face) bounding-box walk; 64-bit (depth key | face id)
//                   atomicMin into the visibility buffer               (.cu:184-255)
//   k_resolve       one thread per pixel: decode the winner, recompute its barycentrics,
//                   shade, write all pixel outputs, reset the visibility key (.cu:74-91,262-408)
//   k_normal_map    texel-space normal map                             (.cu:415-445)
#include <algorithm>

#include "gvv_kernels.hpp"
#include "gvv_raster.hpp"
#include "gvv_shade.hpp"

namespace gvv {

// The setup stages of one call as one launch (SetupArgs): blocks [0, cb) set up cameras (block
// 0 also clears the large-face counters), blocks [cb, cb + fb) set up faces, and the rest
// zero-fill the listed buffers, 16 bytes per lane where a buffer is 16-byte aligned.
__device__ __forceinline__ void setup_body(const SetupGrid& g, int blk) {
  const SetupArgs& a = g.a;
  const int t = threadIdx.x;
  if (blk < g.cam_blocks) {
    if (blk == 0 && a.counters && t < 2) a.counters[t] = 0u;
    const int i = blk * 256 + t;
    if (i < a.n_cams) {
      Camera c;
      camera_setup(a.extr + 12 * (size_t)i, a.intr + 9 * (size_t)i, c);
      a.cams[i] = c;
      if (a.view_err) a.view_err[i] = view_error(c, a.W, a.H);
    }
    return;
  }
  blk -= g.cam_blocks;
  if (blk < g.face_blocks) {
    const int64_t i = (int64_t)blk * 256 + t;
    if (i >= (int64_t)a.B * a.F) return;
    const int b = (int)(i / a.F), f = (int)(i % a.F);
    const float* vp = a.vpos + (size_t)b * a.N * 3;
    const V3 v0 = ld3(vp + 3 * a.faces[3 * f]), v1 = ld3(vp + 3 * a.faces[3 * f + 1]),
             v2 = ld3(vp + 3 * a.faces[3 * f + 2]);
    if (a.fnormal) {
      const V3 n = cross(v1 - v0, v2 - v0);
      float* o = a.fnormal + 3 * i;
      o[0] = n.x; o[1] = n.y; o[2] = n.z;
    }
    if (a.tris) {
      TriSetup t = tri_setup(v0, v1, v2);
      t.shape = face_shape(t);
      a.tris[i] = t;
    }
    if (a.face_grad) {
      FaceGrad r;
      r.t = tri_setup(v0, v1, v2);
      r.g = bary_face_setup(v0, v1, v2);
      a.face_grad[i] = r;
    }
    return;
  }
  blk -= g.face_blocks;
  const int64_t start = (int64_t)blk * 256 + t, stride = (int64_t)g.fill_blocks * 256;
  for (int k = 0; k < kFillSegs; ++k) {
    float* p = a.fill[k];
    const int64_t n = a.fill_n[k];
    if (!p || n <= 0) continue;
    int64_t head = 0;
    if (((uintptr_t)p & 15) == 0) {
      const int64_t n4 = n >> 2;
      float4* p4 = reinterpret_cast<float4*>(p);
      for (int64_t i = start; i < n4; i += stride) p4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      head = n4 << 2;
    }
    for (int64_t i = head + start; i < n; i += stride) p[i] = 0.f;
  }
}

__global__ void __launch_bounds__(256) k_setup(SetupGrid g) { setup_body(g, blockIdx.x); }

__global__ void __launch_bounds__(256) k_setup_multi(MeshTable<SetupGrid> t) {
  const MeshSlice m = t.find(blockIdx.x);
  const SetupGrid g = t.load(m.mesh);
  setup_body(g, (int)m.local);
}

// One thread per (b, c, vertex): vertex normal as the CSR-ordered sum of incident face
// normals (first term assigned, the rest added), written per view; projection into view c.
// `blk` is the mesh's own 256-thread block index.
__device__ __forceinline__ void vertices_body(const VertexArgs& va, int64_t blk) {
  const float* __restrict__ vpos = va.vpos;
  const float* __restrict__ fnormal = va.fnormal;
  const int32_t* __restrict__ csr_start = va.csr_start;
  const int32_t* __restrict__ csr_count = va.csr_count;
  const int32_t* __restrict__ csr_list = va.csr_list;
  const Camera* __restrict__ cams = va.cams;
  float* __restrict__ vnormal = va.vnormal;
  float4* __restrict__ proj = va.proj;
  const int B = va.B, C = va.C, N = va.N, F = va.F;
  // one thread per (view, vertex)
  const int64_t i = blk * 256 + threadIdx.x;
  const bool valid = i < (int64_t)B * C * N;
  const int v = valid ? (int)(i % N) : 0;
  const int bc = valid ? (int)(i / N) : 0;
  const int b = bc / C;
  const float* fn = fnormal + (size_t)b * F * 3;
  const int s = valid ? csr_start[v] : 0, n = valid ? csr_count[v] : 0;
  // Vertices of up to kHeavy incident faces sum them in their own lane, loading the face ids
  // and then the normals of kBatch faces at a time.  More incident faces (the centre of a fan:
  // hundreds) would make one lane's chain of loads the whole kernel's time, so the wavefront
  // loads their normals 64 at a time and folds them in list order with readlane.  Both keep
  // the reference's summation order.
  constexpr int kBatch = 8, kHeavy = 2 * kBatch;
  V3 acc = v3(0.f, 0.f, 0.f);
  if (n <= kHeavy) {
    for (int k0 = 0; k0 < n; k0 += kBatch) {
      int id[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) id[j] = k0 + j < n ? csr_list[s + k0 + j] : 0;
      V3 q[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) q[j] = k0 + j < n ? ld3(fn + 3 * id[j]) : v3(0.f, 0.f, 0.f);
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        if (k0 + j >= n) break;
        if (k0 + j == 0) acc = q[j];
        else { acc.x = acc.x + q[j].x; acc.y = acc.y + q[j].y; acc.z = acc.z + q[j].z; }
      }
    }
  }
  const int lane = threadIdx.x & 63;
  __shared__ float s_fold[4][64 * 3];   // one row per wavefront of the 256-thread workgroup
  float* fold = s_fold[threadIdx.x >> 6];
  for (uint64_t heavy = __ballot(n > kHeavy); heavy; heavy &= heavy - 1) {
    const int j = __ffsll((unsigned long long)heavy) - 1;
    const int sj = __builtin_amdgcn_readlane(s, j), nj = __builtin_amdgcn_readlane(n, j);
    const float* fnj = fnormal + (size_t)__builtin_amdgcn_readlane(b, j) * F * 3;
    V3 sum = v3(0.f, 0.f, 0.f);
    // 256 entries per pass: the face ids of all four 64-entry chunks, then their normals, are
    // loaded at once (entries past the end repeat the last and are not summed), then folded
    for (int k0 = 0; k0 < nj; k0 += 256) {
      int id[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) id[c] = csr_list[sj + min(k0 + 64 * c + lane, nj - 1)];
      V3 q[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) q[c] = ld3(fnj + 3 * id[c]);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int cnt = min(64, nj - (k0 + 64 * c));
        if (cnt <= 0) break;
        // the chunk goes through this wavefront's LDS row and every lane folds it in list
        // order from there (uniform-address reads pipeline; a readlane per value does not)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        fold[3 * lane + 0] = q[c].x; fold[3 * lane + 1] = q[c].y; fold[3 * lane + 2] = q[c].z;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 8
        for (int t = 0; t < cnt; ++t) {
          const float qx = fold[3 * t], qy = fold[3 * t + 1], qz = fold[3 * t + 2];
          if (k0 + 64 * c + t == 0) sum = v3(qx, qy, qz);
          else { sum.x = sum.x + qx; sum.y = sum.y + qy; sum.z = sum.z + qz; }
        }
      }
    }
    if (lane == j) acc = sum;
  }
  if (!valid) return;
  float* o = vnormal + 3 * i;
  o[0] = acc.x; o[1] = acc.y; o[2] = acc.z;
  const V3 x = ld3(vpos + ((size_t)b * N + v) * 3);
  const V3 p = project(cams[bc], x);
  proj[i] = make_float4(p.x, p.y, p.z, vertex_error(va.view_err[bc], x, p));
}

__global__ void __launch_bounds__(256) k_vertices(VertexArgs va) { vertices_body(va, blockIdx.x); }

// The multi-mesh kernels copy the mesh's arguments out of the table first, so that they stay in
// scalar registers across the kernel's stores.
__global__ void __launch_bounds__(256) k_vertices_multi(MeshTable<VertexArgs> t) {
  const MeshSlice m = t.find(blockIdx.x);
  const VertexArgs a = t.load(m.mesh);
  vertices_body(a, m.local);
}

constexpr unsigned kLargeWaves = 8192;           // persistent wavefronts of the large-face pass
constexpr unsigned kLargeItems = 8192;          // face parts that a short queue is split into
constexpr int kLargePart = 512;                   // box pixels below which a large face is not split further

struct RasterFace {
  int f, i0, i1, i2;
  float4 p0, p1, p2;
  Box bx;
};

__device__ __forceinline__ RasterFace load_face(const int32_t* __restrict__ faces, const float4* __restrict__ pc,
                                                int f, int W, int H) {
  RasterFace r;
  r.f = f;
  r.i0 = faces[3 * f]; r.i1 = faces[3 * f + 1]; r.i2 = faces[3 * f + 2];
  r.p0 = pc[r.i0]; r.p1 = pc[r.i1]; r.p2 = pc[r.i2];
  r.bx = face_box(v3(r.p0.x, r.p0.y, r.p0.z), v3(r.p1.x, r.p1.y, r.p1.z), v3(r.p2.x, r.p2.y, r.p2.z), W, H);
  return r;
}

// Per-face constants of the exact test, staged in LDS for the candidate pass: the scaled vertices
// and face normal of the ray/triangle test (TriSetup), v0.N - o.N for the face's view, the face id,
// and the binary64 reciprocals of N.N and of the projected depths, which take a 14-cycle product
// for each of the test's five divisions by them in the place of a 45-cycle division (quot).
struct alignas(8) FaceStage {
  float v[12];
  float num;
  int f;
  double rden;
  DepthRecip rz;
};
static_assert(sizeof(FaceStage) == 88, "staged face");

__device__ __forceinline__ void stage_face(FaceStage* dst, const TriSetup& t, V3 os, int f, float z0, float z1, float z2) {
  const float v[12] = {t.v0.x, t.v0.y, t.v0.z, t.v1.x, t.v1.y, t.v1.z, t.v2.x, t.v2.y, t.v2.z, t.N.x, t.N.y, t.N.z};
#pragma unroll
  for (int k = 0; k < 12; ++k) dst->v[k] = v[k];
  dst->num = t.dv0N - dot(os, t.N);
  dst->f = f;
  dst->rden = t.rden;
  dst->rz = depth_recip(z0, z1, z2);
}

// Registers of the face a lane staged (its staging slot is that lane), read by the lanes that
// test its candidates with a cross-lane permute (G lanes hold a face: the first is slot * G).
// The large-face pass holds its one face in every lane.
struct StageOwner {
  int bc, x0, y0, bw;
};

// Candidate list of one wavefront: 32-bit words naming a staged face (its slot) and a pixel.
// Images up to 8192 px on a side pack the pixel itself (slot << 26 | v << 13 | u); larger ones
// keep (slot << 24 | dy * bw + dx) within the face's box, where the depth pass's boxes stay
// below 2^24 px (large_box <= 2^20) and the large-face pass, whose one face is slot 0, gives
// all 32 bits to the box index.
constexpr int kCandCap = 256;        // depth pass
constexpr int kCandCapLarge = 512;   // large-face pass (one staged face, LDS is not the limit)
__device__ __forceinline__ bool cand_packed(int W, int H) { return W <= 8192 && H <= 8192; }
__device__ __forceinline__ unsigned cand_word(bool packed, bool single, int slot, int u, int v, int dx, int dy,
                                              int bw) {
  if (packed) return ((unsigned)slot << 26) | ((unsigned)v << 13) | (unsigned)u;
  const unsigned p = (unsigned)dy * (unsigned)bw + (unsigned)dx;
  return single ? p : (((unsigned)slot << 24) | p);
}

// Exact test of every staged candidate (reference uv2barycentric + inside test + depth key,
// CUDABasedRasterization.cu:237-250), then the 64-bit minimum into the visibility buffer.
// Each lane takes candidates lane, lane+64, ...; all lanes run the expensive test together.
// `single`: the candidates of the large-face pass, which stages one face (slot 0).  Called in
// wave-uniform control flow: the owner reads need every lane active.
template <int G>
__device__ __forceinline__ void flush_candidates(const FaceStage* st, const StageOwner& own, const unsigned* cand,
                                                 int count, const Camera* __restrict__ cams, bool one_view, int bc0,
                                                 unsigned long long* __restrict__ keys, int W, int H, bool single,
                                                 TileMarks marks = TileMarks{}) {
  const int lane = threadIdx.x & 63;
  const bool packed = cand_packed(W, H);
  for (int base = 0; base < count; base += 64) {
    const int i = base + lane;
    const bool valid = i < count;
    const unsigned c = valid ? cand[i] : 0u;
    int slot, u, v;
    if (packed) {
      slot = single ? 0 : (int)(c >> 26);
      v = (int)((c >> 13) & 0x1fffu);
      u = (int)(c & 0x1fffu);
    } else {
      slot = single ? 0 : (int)(c >> 24);
      const unsigned p = single ? c : (c & 0xffffffu);
      const int x0 = __shfl(own.x0, slot * G, 64), y0 = __shfl(own.y0, slot * G, 64);
      const unsigned w = (unsigned)__shfl(own.bw, slot * G, 64);
      const unsigned dy = valid ? p / w : 0u;
      u = x0 + (int)(p - dy * w);
      v = y0 + (int)dy;
    }
    const int bc = one_view ? bc0 : __shfl(own.bc, slot * G, 64);
    if (!valid) continue;
    const FaceStage& fs = st[slot];
    const Camera& cam = cams[bc];
    const V3 d = pixel_ray(cam, u + 0.5f, v + 0.5f);
    TriSetup t;
    t.v0 = v3(fs.v[0], fs.v[1], fs.v[2]);
    t.v1 = v3(fs.v[3], fs.v[4], fs.v[5]);
    t.v2 = v3(fs.v[6], fs.v[7], fs.v[8]);
    t.N = v3(fs.v[9], fs.v[10], fs.v[11]);
    t.rden = fs.rden;
    V3 abc;
    // a and b of a hit are not negative, so that of inside()'s six bounds these three are left
    if (!ray_hit(t, fs.num, cam_origin_scaled(cam), d, abc) || !(abc.x <= 1.001f) || !(abc.y <= 1.001f) ||
        !(abc.z >= -0.001f))
      continue;
    const uint64_t k = pack_key(depth_key(abc, fs.rz), fs.f);
    atomicMin(keys + ((size_t)bc * H + v) * W + u, (unsigned long long)k);
    // screen-tile depth pass: the tile kernel merges this tile's visibility keys
    if (marks.dirty) marks.dirty[((size_t)bc * marks.tiles_y + (v >> marks.sy)) * marks.tiles_x + (u >> marks.sx)] = 1u;
  }
}

// Pre-test the box of staged face `slot` lane-parallel (64 pixels per round) and append the
// passing pixels to the candidate list; flushes first whenever a round could overflow it.
template <int G>
__device__ __forceinline__ void collect_face(const EdgeTest& et_in, int slot, int x0, int y0, int bw, int bh,
                                             FaceStage* st, const StageOwner& own, unsigned* cand, int& count,
                                             const Camera* __restrict__ cams, bool one_view, int bc0,
                                             unsigned long long* __restrict__ keys, int W, int H) {
  const int lane = threadIdx.x & 63;
  const int area = bw * bh;
  for (int base = 0; base < area; base += 64) {
    if (count > kCandCap - 64) {
      __syncthreads();
      flush_candidates<G>(st, own, cand, count, cams, one_view, bc0, keys, W, H, false);
      __syncthreads();
      count = 0;
    }
    const int p = base + lane;
    bool pass = false;
    int dx = 0, dy = 0;
    if (p < area) {
      dy = p / bw;
      dx = p - dy * bw;
      pass = et_in.pass(x0 + dx + 0.5f, y0 + dy + 0.5f);
    }
    const uint64_t m = __ballot(pass);
    if (pass) {
      const int off = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      cand[count + off] = cand_word(cand_packed(W, H), false, slot, x0 + dx, y0 + dy, dx, dy, bw);
    }
    count += __popcll(m);
  }
}

__device__ __forceinline__ EdgeTest readlane_edges(const EdgeTest& e, int j) {
  EdgeTest r;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    r.a[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e.a[i]), j));
    r.b[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e.b[i]), j));
    r.c[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e.c[i]), j));
  }
  r.on = __builtin_amdgcn_readlane((int)e.on, j) != 0;
  return r;
}

// Boxes up to this many pixels are walked line by line by their own lanes, all faces of the
// wavefront at once (BoxLines); larger staged boxes, which only a raised large-face threshold
// brings here, are walked by the whole wavefront, one face at a time.
constexpr int kLineBox = 256;

// Inclusive sum over the 64 lanes (DPP: shifts within the rows of 16, then row broadcasts).
__device__ __forceinline__ int wave_inclusive_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2, 3
  return x;
}

// Appends every lane's span (rem candidates: word, word + step, ...) to the wavefront's list of
// CAP candidates, each span in one piece in lane order; a full list (a multiple of 64) is handed
// to flush() and starts again.  total: the sum of rem over the lanes, incl its inclusive prefix.
template <int CAP, class Flush>
__device__ __forceinline__ void append_spans(unsigned* cand, int& count, int rem, int incl, int total, unsigned word,
                                             unsigned step, Flush&& flush) {
  int pos = count + incl - rem;
  for (;;) {
    for (; rem > 0 && pos < CAP; --rem, ++pos, word += step) cand[pos] = word;
    if (count + total <= CAP) break;
    wave_sync();
    flush(CAP);
    wave_sync();
    total -= CAP - count;
    pos -= CAP;
    count = 0;
  }
  count += total;
}

// One wavefront per 64 / G consecutive (b, c, face) items, G lanes to a face (wg: the mesh's own
// logical block).  Faces with bounding boxes up to large_box pixels are staged and rasterised
// here (line spans, compaction, exact test); larger ones are appended to `large` for
// k_raster_large.
// The G lanes of a face take its lines in turn.  On every step each lane finds the span of its
// line, a wave sum of the span lengths gives each lane its place in the candidate list, and the
// lanes write their spans there; a full list (always a multiple of 64) is tested and emptied.
// The spans replace an edge test of every box pixel, one pixel of 64 boxes per step with 13.75 of
// the 64 lanes passing on average at 100k triangles over 8 x 1024^2 views: 249 -> 153 us there.
// What bounds it now, there, is the memory side's rate of atomic requests, 2.24 M in 113 us, 20 G/s
// of the 21 G/s that scattered atomics reach (the large-face pass 0.50 M in 31 us, 16 G/s), and
// VALU issue at 83% (57 M instructions).  Reading a pixel's key before the exact test, to skip the
// atomic where the face cannot win, adds a memory-side request for each it saves: 165 us.
// Appends the lanes' faces with `large` set to the large-face queue, with one atomic per wavefront.
__device__ __forceinline__ void queue_large(const RasterArgs& ra, bool large, int bc, int f) {
  const uint64_t qm = __ballot(large);
  if (!qm) return;
  unsigned int base = 0;
  if ((int)(threadIdx.x & 63) == __ffsll((unsigned long long)qm) - 1) base = atomicAdd(ra.large_count, (unsigned)__popcll(qm));
  base = __builtin_amdgcn_readlane(base, __ffsll((unsigned long long)qm) - 1);
  if (large) {
    const unsigned off = __builtin_amdgcn_mbcnt_hi((unsigned)(qm >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)qm, 0u));
    ra.large[base + off] = make_int4(bc, f, ra.mesh_id, 0);
  }
}

template <int G>
__device__ __forceinline__ void raster_body(const RasterArgs& ra, int64_t wg) {
  constexpr int kFaces = 64 / G;
  const TriSetup* __restrict__ tris = ra.tris;
  const int32_t* __restrict__ faces = ra.faces;
  const float4* __restrict__ proj = ra.proj;
  const Camera* __restrict__ cams = ra.cams;
  unsigned long long* __restrict__ keys = ra.keys;
  const int B = ra.B, C = ra.C, N = ra.N, F = ra.F, W = ra.W, H = ra.H, large_box = ra.large_box;
  __shared__ FaceStage st[kFaces];
  __shared__ unsigned cand[kCandCap];
  const int lane = threadIdx.x, slot = lane / G, sub = lane % G;
  const int64_t items = (int64_t)B * C * F;
  // Large faces go to the queue 64 items at a time whatever G: the queue's cursor is one word on the
  // memory side, which takes an atomic each 6 to 11 ns, so with an atomic per wavefront of 4 faces a
  // mesh whose faces are mostly large waited for it (64,000 faces of about 6 x 40 px: 171 us, 31 now;
  // 19,200 of 10 x 70 px 64 and 12).
  // With several lanes to a face every G-th wavefront looks at the boxes of its own and the next
  // G - 1 wavefronts' faces, one lane to a face.
  if (G > 1 && wg % G == 0) {
    const int64_t q = wg * kFaces + lane;
    bool big = false;
    int qf = 0, qbc = 0;
    if (q < items) {
      qf = (int)(q % F);
      qbc = (int)(q / F);
      const Box bx = load_face(faces, proj + (size_t)qbc * N, qf, W, H).bx;
      big = bx.x0 <= bx.x1 && bx.y0 <= bx.y1 && (int64_t)(bx.x1 - bx.x0 + 1) * (bx.y1 - bx.y0 + 1) > large_box;
    }
    queue_large(ra, big, qbc, qf);
  }
  const int64_t i = wg * kFaces + slot;
  const bool in_range = i < items;
  const int f = in_range ? (int)(i % F) : 0;
  const int bc = in_range ? (int)(i / F) : 0;
  bool small = false, to_queue = false;
  EdgeTest et;
  et.on = false;
  for (int k = 0; k < 3; ++k) et.a[k] = et.b[k] = et.c[k] = 0.f;
  int bw = 0, bh = 0, fx0 = 0, fy0 = 0;
  if (in_range) {
    const RasterFace r = load_face(faces, proj + (size_t)bc * N, f, W, H);
    if (r.bx.x0 <= r.bx.x1 && r.bx.y0 <= r.bx.y1) {
      bw = r.bx.x1 - r.bx.x0 + 1;
      bh = r.bx.y1 - r.bx.y0 + 1;
      if ((int64_t)bw * bh > large_box) {
        to_queue = G == 1;
      } else {
        small = true;
        const TriSetup& tri = tris[(size_t)(bc / C) * F + f];
        if (sub == 0) stage_face(&st[slot], tri, cam_origin_scaled(cams[bc]), f, r.p0.z, r.p1.z, r.p2.z);
        et = edge_test(r.p0, r.p1, r.p2, tri.shape, r.bx);
        fx0 = r.bx.x0;
        fy0 = r.bx.y0;
      }
    }
  }
  if (G == 1) queue_large(ra, to_queue, bc, f);
  if (!__ballot(small)) return;
  const int bc0 = __builtin_amdgcn_readfirstlane(bc);
  const bool one_view = __ballot(bc != bc0 && in_range) == 0;
  const StageOwner own{bc, fx0, fy0, bw};
  __syncthreads();
  int count = 0;
  const bool packed = cand_packed(W, H);
  const bool by_line = small && bw * bh <= kLineBox;
  BoxLines bl;
  bl.start(et, fx0, fy0, bw, bh);
  const int lines = by_line ? bl.lines : 0;
  const unsigned step = cand_word(packed, false, 0, bl.columns ? 0 : 1, bl.columns ? 1 : 0, bl.columns ? 0 : 1,
                                  bl.columns ? 1 : 0, bw);
  for (int ln = sub; __ballot(ln < lines); ln += G) {
    int first = 0;
    const int rem = ln < lines ? bl.span(ln, first) : 0;
    const int incl = wave_inclusive_sum(rem);
    const int dx = bl.columns ? ln : first, dy = bl.columns ? first : ln;
    const unsigned word = cand_word(packed, false, slot, fx0 + dx, fy0 + dy, dx, dy, bw);
    append_spans<kCandCap>(cand, count, rem, incl, __builtin_amdgcn_readlane(incl, 63), word, step, [&](int n) {
      flush_candidates<G>(st, own, cand, n, cams, one_view, bc0, keys, W, H, false);
    });
  }
  // larger staged boxes: the whole wavefront walks one box at a time
  uint64_t todo = __ballot(small && !by_line && sub == 0);
  while (todo) {
    const int j = __ffsll((unsigned long long)todo) - 1;
    todo &= todo - 1;
    const EdgeTest ej = readlane_edges(et, j);
    const int x0 = __builtin_amdgcn_readlane(fx0, j), y0 = __builtin_amdgcn_readlane(fy0, j);
    const int jbw = __builtin_amdgcn_readlane(bw, j), jbh = __builtin_amdgcn_readlane(bh, j);
    collect_face<G>(ej, j / G, x0, y0, jbw, jbh, st, own, cand, count, cams, one_view, bc0, keys, W, H);
  }
  __syncthreads();
  flush_candidates<G>(st, own, cand, count, cams, one_view, bc0, keys, W, H, false);
}

template <int G>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8))) k_raster(RasterArgs ra) {
  raster_body<G>(ra, xcd_contiguous(blockIdx.x, gridDim.x));
}

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8))) k_raster_multi(MeshTable<RasterArgs> t) {
  const MeshSlice m = t.find((unsigned)xcd_contiguous(blockIdx.x, gridDim.x));
  const RasterArgs a = t.load(m.mesh);
  raster_body<kBatchedLanes>(a, m.local);
}

// Part `part` of `parts` of one large face (bc, f), rasterised by the whole wavefront: rows part,
// part + parts, ... of its box.  The spans of 64 rows are found at once, one per lane
// (BoxLines).  They go to the candidate list one span at a time, 64 pixels per step, or, where
// they are shorter than they are many (a sliver across its box), all at once, one pixel of each
// per step.  Full lists take the exact test as in k_raster.
// Rows also of tall boxes: the pass is bound by the memory side's atomic requests, one per 64-byte line
// of keys and instruction, and 64 candidates along a column are 64 lines.  With the columns of tall
// boxes it took 341 us at 2,400 tall faces (about 10 x 70 px) over 8 x 1024^2 and takes 141 with rows,
// 146 -> 65 us at 320 faces over 4 x 1024^2.
__device__ __forceinline__ void raster_large_face(const TriSetup* __restrict__ tris, const int32_t* __restrict__ faces,
                                                  const float4* __restrict__ proj, const Camera* __restrict__ cams,
                                                  unsigned long long* __restrict__ keys, int C, int N, int F, int W,
                                                  int H, int bc, int f, int part, int parts, FaceStage* st,
                                                  unsigned* cand, TileMarks marks) {
  const RasterFace r = load_face(faces, proj + (size_t)bc * N, f, W, H);
  const int bw = r.bx.x1 - r.bx.x0 + 1, bh = r.bx.y1 - r.bx.y0 + 1;
  parts = max(1, min(parts, min(bh, (int)(((int64_t)bw * bh) / kLargePart))));
  if (part >= parts) return;
  const TriSetup& tri = tris[(size_t)(bc / C) * F + f];
  BoxLines bl;
  bl.start_rows(edge_test(r.p0, r.p1, r.p2, tri.shape, r.bx), r.bx.x0, r.bx.y0, bw, bh);
  const int lane = threadIdx.x & 63;
  wave_sync();
  if (lane == 0) stage_face(&st[0], tri, cam_origin_scaled(cams[bc]), f, r.p0.z, r.p1.z, r.p2.z);
  const StageOwner own{bc, r.bx.x0, r.bx.y0, bw};
  wave_sync();
  const bool packed = cand_packed(W, H);
  const unsigned step = cand_word(packed, true, 0, 1, 0, 1, 0, bw);
  int count = 0;
  const auto flush = [&](int n) {
    flush_candidates<1>(st, own, cand, n, cams, true, bc, keys, W, H, true, marks);
  };
  for (int l0 = part; l0 < bl.lines; l0 += 64 * parts) {
    const int ln = l0 + lane * parts;
    int first = 0;
    const int len = ln < bl.lines ? bl.span(ln, first) : 0;
    const unsigned word = cand_word(packed, true, 0, r.bx.x0 + first, r.bx.y0 + ln, first, ln, bw);
    uint64_t todo = __ballot(len > 0);
    const int incl = wave_inclusive_sum(len), total = __builtin_amdgcn_readlane(incl, 63), spans = __popcll(todo);
    if (2 * total <= spans * spans) {
      append_spans<kCandCapLarge>(cand, count, len, incl, total, word, step, flush);
      continue;
    }
    for (; todo; todo &= todo - 1) {
      const int j = __ffsll((unsigned long long)todo) - 1;
      const unsigned word_j = __builtin_amdgcn_readlane(word, j);
      const int len_j = __builtin_amdgcn_readlane(len, j);
      for (int k0 = 0; k0 < len_j; k0 += 64) {
        if (count > kCandCapLarge - 64) {
          wave_sync();
          flush(count);
          wave_sync();
          count = 0;
        }
        if (k0 + lane < len_j) cand[count + lane] = word_j + (unsigned)(k0 + lane) * step;
        count += min(64, len_j - k0);
      }
    }
  }
  wave_sync();
  flush(count);
}

// Persistent wavefronts drain the large-face queue, whose length k_raster wrote: n faces are split
// into kLargeItems / n parts each (at least one; a face of few pixels is split less), and of G
// wavefronts, w takes parts w, w + G, ...  A shared atomic cursor would balance better, but every
// wavefront taking every item from one word serialises on that word's memory-side atomics: 4k
// cursor atomics took longer than the faces themselves.
// A part repeats the face's setup (about 300 instructions) but no pixel's work, so that a short
// queue fills the chip: 1,280 faces of about 3,000 px each took 373 us with one wavefront per
// face.  The pass follows k_raster on the same stream: beside it, on a second stream with a
// kernel of its own to fill the queue, the fork and join left 6 and 10 us of idle time per
// forward, as much as the overlap saved (100k faces over 8 x 1024^2: 651 us forward + backward
// beside, 662 in line; 304 against 278 for the 1,280 faces, 173 against 161 for 6 x 333 x 477).
__device__ __forceinline__ int large_parts(unsigned n_large) {
  return (int)min(max(kLargeItems / max(n_large, 1u), 1u), 64u);
}

__global__ void __launch_bounds__(64) k_raster_large(const TriSetup* __restrict__ tris, const int32_t* __restrict__ faces,
                                                     const float4* __restrict__ proj, const Camera* __restrict__ cams,
                                                     unsigned long long* __restrict__ keys,
                                                     unsigned int* __restrict__ counters, const int4* __restrict__ large,
                                                     int C, int N, int F, int W, int H, TileMarks marks) {
  __shared__ FaceStage st[1];
  __shared__ unsigned cand[kCandCapLarge];
  const unsigned int n_large = counters[0];
  const unsigned int parts = (unsigned)large_parts(n_large);
  for (unsigned int item = blockIdx.x; item < n_large * parts; item += gridDim.x) {
    const int4 e = large[item / parts];
    raster_large_face(tris, faces, proj, cams, keys, C, N, F, W, H, e.x, e.y, (int)(item % parts), (int)parts, st, cand,
                      marks);
  }
}

// The same over a queue shared by several meshes: each entry names its mesh, whose raster
// state comes from the descriptor table.  One launch drains the large faces of every mesh.
__global__ void __launch_bounds__(64) k_raster_large_multi(const RasterMesh* __restrict__ meshes,
                                                           unsigned int* __restrict__ counters,
                                                           const int4* __restrict__ large) {
  __shared__ FaceStage st[1];
  __shared__ unsigned cand[kCandCapLarge];
  const unsigned int n_large = counters[0];
  const unsigned int parts = (unsigned)large_parts(n_large);
  for (unsigned int item = blockIdx.x; item < n_large * parts; item += gridDim.x) {
    const int4 e = large[item / parts];
    const RasterMesh m = meshes[e.z];
    raster_large_face(m.tris, m.faces, m.proj, m.cams, m.keys, m.C, m.N, m.F, m.W, m.H, e.x, e.y, (int)(item % parts),
                      (int)parts, st, cand, m.marks);
  }
}

__global__ void k_zero_u32(unsigned int* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0u;
}

template <int ALBEDO, bool SHADE>
__device__ __forceinline__ void resolve_body(const ResolveArgs& a, unsigned wg) {
  // one workgroup per 256-pixel chunk of one image row: the view, row and chunk follow from the
  // workgroup index alone (uniform arithmetic), so no lane divides its pixel index
  const unsigned chunks = ((unsigned)a.W + 255u) >> 8;
  const unsigned per_view = chunks * (unsigned)a.H;
  const int bc = (int)(wg / per_view);
  const unsigned rem = wg - (unsigned)bc * per_view;
  const int py = (int)(rem / chunks);
  const int px = (int)(rem - (unsigned)py * chunks) * 256 + (int)threadIdx.x;
  if (bc >= a.B * a.C || px >= a.W) return;
  const int64_t i = ((int64_t)bc * a.H + py) * a.W + px;
  unsigned long long key = a.keys[i];
  if (key == kEmptyKey) {
    background_pixel(a, i);
    return;
  }
  st_out(a.keys + i, (unsigned long long)kEmptyKey);   // next read by the next call's depth pass
  shade_pixel<ALBEDO, SHADE>(a, bc, i, (int)(uint32_t)(key & 0xffffffffu), pixel_ray(a.cams[bc], px + 0.5f, py + 0.5f));
}

template <int ALBEDO, bool SHADE>
__global__ void __launch_bounds__(256) k_resolve(ResolveArgs a) {
  resolve_body<ALBEDO, SHADE>(a, (unsigned)xcd_contiguous(blockIdx.x, gridDim.x));
}

template <int ALBEDO, bool SHADE>
__global__ void __launch_bounds__(256) k_resolve_multi(MeshTable<ResolveArgs> t) {
  const MeshSlice m = t.find((unsigned)xcd_contiguous(blockIdx.x, gridDim.x));
  const ResolveArgs a = t.load(m.mesh);
  resolve_body<ALBEDO, SHADE>(a, (unsigned)m.local);
}

__global__ void __launch_bounds__(256) k_normal_map(const UvTexel* __restrict__ table, const int32_t* __restrict__ faces,
                                                    const float* __restrict__ vnormal, float* __restrict__ nmap,
                                                    int B, int C, int N, int T) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)B * T) return;
  int b = (int)(i / T), t = (int)(i % T);
  UvTexel e = table[t];
  const float* vn = vnormal + (size_t)b * C * N * 3;   // view 0
  int f = e.face;
  V3 n = ld3(vn + 3 * faces[3 * f]) * e.a + ld3(vn + 3 * faces[3 * f + 1]) * e.b + ld3(vn + 3 * faces[3 * f + 2]) * e.c;
  float len = length(n);
  if (len != 0.f) n = n / len;
  float* o = nmap + 3 * i;
  o[0] = (n.x + 1.f) / 2.f; o[1] = (n.y + 1.f) / 2.f; o[2] = (n.z + 1.f) / 2.f;
}

__global__ void __launch_bounds__(256) k_fill_u64(unsigned long long* p, int64_t n, unsigned long long v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void __launch_bounds__(256) k_fill_f32(float* p, int64_t n, float v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ------------------------------------------------------------------------------------------
// host-side launchers
// ------------------------------------------------------------------------------------------
static inline unsigned blocks_for(int64_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }

hipError_t launch_fill_u64(unsigned long long* p, int64_t n, unsigned long long v, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u64, dim3(blocks_for(n)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_fill_f32(float* p, int64_t n, float v, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_f32, dim3(blocks_for(n)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

SetupGrid setup_grid(const SetupArgs& a) {
  SetupGrid g;
  g.a = a;
  g.cam_blocks = a.n_cams > 0 || a.counters ? (int)blocks_for(a.n_cams > 0 ? a.n_cams : 1) : 0;
  g.face_blocks = a.faces ? (int)blocks_for((int64_t)a.B * a.F) : 0;
  int64_t most = 0;
  for (int k = 0; k < kFillSegs; ++k)
    if (a.fill[k] && a.fill_n[k] > most) most = a.fill_n[k];
  g.fill_blocks = most > 0 ? (int)std::min<int64_t>(2048, (int64_t)blocks_for((most + 3) / 4)) : 0;
  return g;
}

hipError_t launch_setup(const SetupArgs& a, hipStream_t s) {
  const SetupGrid g = setup_grid(a);
  const int total = g.cam_blocks + g.face_blocks + g.fill_blocks;
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL(k_setup, dim3(total), dim3(256), 0, s, g);
  return hipGetLastError();
}

template <int ALBEDO, bool SHADE>
static void launch_resolve_t(const ResolveArgs& a, hipStream_t s) {
  const int64_t n = (int64_t)a.B * a.C * a.H * ((a.W + 255) / 256);   // workgroups: row chunks
  if (n <= 0) return;
  hipLaunchKernelGGL((k_resolve<ALBEDO, SHADE>), dim3((unsigned)n), dim3(256), 0, s, a);
}

SetupArgs forward_setup_args(const ForwardPlan& p) {
  SetupArgs sa;
  sa.extr = p.extr; sa.intr = p.intr; sa.cams = p.cams; sa.n_cams = p.B * p.C;
  sa.view_err = p.view_err; sa.W = p.r.W; sa.H = p.r.H;
  sa.vpos = p.vpos; sa.faces = p.faces; sa.fnormal = p.fnormal; sa.tris = p.tris;
  sa.B = p.B; sa.N = p.N; sa.F = p.F;
  sa.counters = p.shared_queue ? nullptr : p.counters;
  return sa;
}

VertexArgs vertex_args(const ForwardPlan& p) {
  VertexArgs a;
  a.vpos = p.vpos; a.fnormal = p.fnormal; a.csr_start = p.csr_start; a.csr_count = p.csr_count;
  a.csr_list = p.csr_list; a.cams = p.cams; a.view_err = p.view_err; a.vnormal = p.vnormal_out; a.proj = p.proj;
  a.B = p.B; a.C = p.C; a.N = p.N; a.F = p.F;
  return a;
}

RasterArgs raster_args(const ForwardPlan& p) {
  RasterArgs a;
  a.tris = p.tris; a.faces = p.faces; a.proj = p.proj; a.cams = p.cams; a.keys = p.r.keys;
  a.large_count = p.counters; a.large = p.large;
  a.B = p.B; a.C = p.C; a.N = p.N; a.F = p.F; a.W = p.r.W; a.H = p.r.H;
  a.large_box = p.large_box; a.mesh_id = p.mesh_id;
  return a;
}

RasterMesh raster_mesh(const ForwardPlan& p) {
  RasterMesh m;
  m.tris = p.tris; m.faces = p.faces; m.proj = p.proj; m.cams = p.cams; m.keys = p.r.keys;
  m.C = p.C; m.N = p.N; m.F = p.F; m.W = p.r.W; m.H = p.r.H;
  m.marks = p.tiled ? p.marks : TileMarks{};
  return m;
}

hipError_t launch_clear_counters(unsigned int* counters, hipStream_t s) {
  hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, counters, 2);
  return hipGetLastError();
}

hipError_t launch_raster_large_multi(const RasterMesh* meshes, unsigned int* counters, const int4* large,
                                     hipStream_t s) {
  hipLaunchKernelGGL(k_raster_large_multi, dim3(kLargeWaves), dim3(64), 0, s, meshes, counters, large);
  return hipGetLastError();
}

static void launch_raster(const ForwardPlan& p, const RasterArgs& ra, hipStream_t s) {
  const int64_t items = (int64_t)ra.B * ra.C * ra.F;
  const int g = raster_lanes(p.raster_items);
  const dim3 grid(blocks_for(items, 64 / g));
  if (g == 16) hipLaunchKernelGGL(k_raster<16>, grid, dim3(64), 0, s, ra);
  else if (g == 8) hipLaunchKernelGGL(k_raster<8>, grid, dim3(64), 0, s, ra);
  else if (g == 2) hipLaunchKernelGGL(k_raster<2>, grid, dim3(64), 0, s, ra);
  else hipLaunchKernelGGL(k_raster<1>, grid, dim3(64), 0, s, ra);
}

hipError_t launch_forward_raster(const ForwardPlan& p, hipStream_t s) {
  const int B = p.B, C = p.C, N = p.N, F = p.F;
  {
    // cameras, face setup and (for a queue of its own) the large-face counters
    ProfScope ps(p.prof, "k_setup", s);
    hipError_t e = launch_setup(forward_setup_args(p), s);
    if (e != hipSuccess) return e;
  }
  {
    ProfScope ps(p.prof, "k_vertices", s);
    hipLaunchKernelGGL(k_vertices, dim3(blocks_for((int64_t)B * C * N)), dim3(256), 0, s, vertex_args(p));
  }
  if (p.normal_map) {
    ProfScope ps(p.prof, "k_normal_map", s);
    int T = p.r.texW * p.r.texH;
    hipLaunchKernelGGL(k_normal_map, dim3(blocks_for((int64_t)B * T)), dim3(256), 0, s, p.uv_table, p.faces,
                       p.vnormal_out, p.normal_map_out, B, C, N, T);
    return hipGetLastError();
  }
  if (p.tiled) {
    ProfScope ps(p.prof, "k_bin", s);
    hipError_t e = launch_bin(p, s);
    if (e != hipSuccess) return e;
  } else {
    ProfScope ps(p.prof, "k_raster", s);
    launch_raster(p, raster_args(p), s);
  }
  if (!p.shared_queue) {
    ProfScope ps(p.prof, "k_raster_large", s);
    hipLaunchKernelGGL(k_raster_large, dim3(kLargeWaves), dim3(64), 0, s, p.tris, p.faces, p.proj, p.cams,
                       p.r.keys, p.counters, p.large, C, N, F, p.r.W, p.r.H, p.tiled ? p.marks : TileMarks{});
  }
  return hipGetLastError();
}

hipError_t launch_forward_resolve(const ForwardPlan& p, hipStream_t s) {
  // In normal-map mode the visibility buffer is empty, so this writes the background.
  // One workgroup per 256-pixel row chunk: the count must fit a 32-bit grid dimension.
  if (p.tiled && !p.normal_map) {
    ProfScope ps(p.prof, "k_tile", s);
    return launch_tile(p, s);
  }
  if ((int64_t)p.r.B * p.r.C * p.r.H * ((p.r.W + 255) / 256) > (int64_t)UINT32_MAX) return hipErrorInvalidConfiguration;
  ProfScope ps(p.prof, "k_resolve", s);
  switch (p.albedo * 2 + (p.shade ? 1 : 0)) {
    case kVertexColor * 2 + 0: launch_resolve_t<kVertexColor, false>(p.r, s); break;
    case kVertexColor * 2 + 1: launch_resolve_t<kVertexColor, true>(p.r, s); break;
    case kTextured * 2 + 0: launch_resolve_t<kTextured, false>(p.r, s); break;
    case kTextured * 2 + 1: launch_resolve_t<kTextured, true>(p.r, s); break;
    case kNormal * 2 + 0: launch_resolve_t<kNormal, false>(p.r, s); break;
    case kNormal * 2 + 1: launch_resolve_t<kNormal, true>(p.r, s); break;
    case kLighting * 2 + 0: launch_resolve_t<kLighting, false>(p.r, s); break;
    case kLighting * 2 + 1: launch_resolve_t<kLighting, true>(p.r, s); break;
    case kForegroundMask * 2 + 0: launch_resolve_t<kForegroundMask, false>(p.r, s); break;
    default: launch_resolve_t<kForegroundMask, true>(p.r, s); break;
  }
  return hipGetLastError();
}

hipError_t launch_setup_multi(const MeshTable<SetupGrid>& t, unsigned blocks, hipStream_t s) {
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_setup_multi, dim3(blocks), dim3(256), 0, s, t);
  return hipGetLastError();
}

hipError_t launch_vertices_multi(const MeshTable<VertexArgs>& t, unsigned blocks, hipStream_t s) {
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_vertices_multi, dim3(blocks), dim3(256), 0, s, t);
  return hipGetLastError();
}

hipError_t launch_raster_multi(const MeshTable<RasterArgs>& t, unsigned blocks, hipStream_t s) {
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_raster_multi, dim3(blocks), dim3(64), 0, s, t);
  return hipGetLastError();
}

hipError_t launch_resolve_multi(const MeshTable<ResolveArgs>& t, unsigned blocks, int albedo, bool shade,
                                hipStream_t s) {
  if (blocks == 0) return hipSuccess;
  switch (albedo * 2 + (shade ? 1 : 0)) {
    case kVertexColor * 2 + 0: hipLaunchKernelGGL((k_resolve_multi<kVertexColor, false>), dim3(blocks), dim3(256), 0, s, t); break;
    case kVertexColor * 2 + 1: hipLaunchKernelGGL((k_resolve_multi<kVertexColor, true>), dim3(blocks), dim3(256), 0, s, t); break;
    case kTextured * 2 + 0: hipLaunchKernelGGL((k_resolve_multi<kTextured, false>), dim3(blocks), dim3(256), 0, s, t); break;
    case kTextured * 2 + 1: hipLaunchKernelGGL((k_resolve_multi<kTextured, true>), dim3(blocks), dim3(256), 0, s, t); break;
    case kForegroundMask * 2 + 0:
      hipLaunchKernelGGL((k_resolve_multi<kForegroundMask, false>), dim3(blocks), dim3(256), 0, s, t);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

unsigned resolve_blocks(const ResolveArgs& a) { return (unsigned)((int64_t)a.B * a.C * a.H * ((a.W + 255) / 256)); }

hipError_t launch_forward(const ForwardPlan& p, hipStream_t s) {
  hipError_t e = launch_forward_raster(p, s);
  if (e != hipSuccess) return e;
  return launch_forward_resolve(p, s);
}

}  // namespace gvv
