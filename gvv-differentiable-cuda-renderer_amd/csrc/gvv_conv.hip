// gvv_conv.hip -- BF16 MFMA convolutions of the proposal network (declared in include/gvv_proposal.h).
//
// The reference has no learned component; these kernels serve the proposal network that
// warm-starts the analysis-by-synthesis fit.  Every convolution (and the linear head, as a
// 1x1 convolution over a 1x1 image) is an implicit GEMM on v_mfma_f32_16x16x32_bf16 with
// FP32 accumulation:
//
//   forward        O[q][p] = sum_k P[p][k] Q[q][k]   p = output channel, q = output pixel,
//                                                    k = (kh, kw, ci)
//   backward data  p = input channel, q = input pixel, k = (kh, kw, co).  Input pixels are taken
//                  by their residue modulo the stride: pixels of one residue class see the same
//                  taps, so only taps on the stride grid are loaded and multiplied
//   backward wt    p = (kh, kw, ci), q = output channel, k = output pixel
//
// Activations are NHWC bf16 with the channel count a multiple of 8, so that 8 consecutive k
// are 8 consecutive channels of one tap: one 16-byte load per MFMA operand chunk.
//
// What bounds these layers is latency: at 16 images of 256^2 the whole network is 7 GFLOP and
// 50 MB forward (6 and 10 us at this card's rates), over layers of 3 to 128 MFMA depths with
// 128 to 4096 output tiles of 64 x 64.  So the loads of one output tile's reduction are shared out
// over the waves of a workgroup: each wave loads the operands of its stretch of k straight from
// global memory into MFMA registers, all at once, with no LDS staging.  Forward and backward data
// keep one accumulation chain per output, in k order, whatever the tile and the number of waves
// (their results feed bf16 roundings, which another order of addition would move): the
// accumulators go from wave to wave through LDS, and each wave adds its stretch when they arrive.
// The chain is short next to the loads it no longer waits for (a step of 32 k is 16 cycles of a
// dependent MFMA).  The weight gradient, an FP32 result, adds the waves' own sums at the end.
// Staging both operands in LDS with two barriers per 32 k took 236 us for the seven forward
// layers of 16 images and 212 us for one, 290 for backward data and 385 for the weights of 16.
//
// MFMA lane layout (16x16x32, wave64): lane l supplies row l%16 of A and column l%16 of B with
// k = 8*(l/16) .. 8*(l/16)+7; it receives D[4*(l/16)+r][l%16] in accumulator r.  A is the P
// side, B the Q side, so each lane ends with 4 consecutive p of one q.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "../../include/gvv_proposal.h"
#include "gvv_kernels.hpp"

namespace gvv {
int set_last_error(const std::string& m);
}

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(uint32_t(h) << 16); }

// float -> bf16, round to nearest even (NaN stays NaN)
__host__ __device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}

struct ConvGeom {
  int B, H, W, Cin, OH, OW, Cout, KS, S, PAD;
};

struct alignas(16) Words4 { uint32_t w[4]; };

__device__ __forceinline__ bf16x8 as_bf16x8(const Words4& v) {
  bf16x8 r;
  __builtin_memcpy(&r, &v, 16);
  return r;
}

// a / b for 0 <= a, b > 0 with a quotient that fits an int: a 32-bit division wherever it can be
__device__ __forceinline__ int quotient(int64_t a, int b) {
  return (a >> 32) == 0 ? int(uint32_t(a) / uint32_t(b)) : int(a / b);
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ---- forward and backward data -----------------------------------------------------------
// One residue class of backward data (forward: the only one): output pixels y = S yc + ry,
// x = S xc + rx; taps kh = kh0 + kstep t, t < nty (kw likewise), reading source row
// (y0 + dir t) with y0 = yc ymul + yadd.
struct Taps {
  int n;                // taps of this axis
  int k0;               // first tap
  int add;              // source position of pixel 0 under the first tap
  int pixels;           // output pixels of this class along the axis
};

__host__ __device__ inline Taps axis_taps(bool fwd, int KS, int S, int PAD, int in, int out, int r) {
  Taps t;
  if (fwd) {
    t.n = KS; t.k0 = 0; t.add = -PAD; t.pixels = out;
  } else {
    t.k0 = (r + PAD) % S;
    t.n = t.k0 < KS ? (KS - t.k0 + S - 1) / S : 0;
    t.add = (r + PAD - t.k0) / S;
    t.pixels = r < in ? (in - r + S - 1) / S : 0;
  }
  return t;
}

struct ConvArgs {
  ConvGeom g;
  const uint16_t* src;     // forward: x [B][H][W][Cin]; backward data: dz [B][OH][OW][Cout]
  const uint16_t* w;       // forward: w [Cout][KS][KS][Cin]; backward data: wt [Cin][KS][KS][Cout]
  const float* bias;       // forward: [Cout]
  const uint16_t* mask;    // backward data: dx *= (mask > 0) where mask is the layer's forward input
  void* out;               // forward: y (bf16 or f32); backward data: dx (bf16)
  int out_f32, relu;
  int wide;                // out and mask are 16-byte aligned
  int ptiles, qtiles;      // tiles of one class
  int classes_x;
};

// 16 TP x 16 TQ outputs per workgroup of NW waves.  The k steps (of 32) are taken in stretches of up
// to NS, wave 0 first; every wave has its next stretch's operands in flight while the accumulators
// travel.
// Few MFMAs go with each operand here, so the integer work around them counts: an output pixel is
// decoded once per row of a tile, and every address is a per-lane pointer plus an offset of the
// step.  ALIGNED (C a multiple of 32): a step lies in one tap, so that offset is uniform and is
// kept in scalar registers; otherwise (the first layer, 8 channels) each 8-channel chunk of a lane
// finds its own tap.
template <bool FWD, bool ALIGNED, int TP, int TQ, int NW, int NS>
__global__ __launch_bounds__(64 * NW) void k_conv(ConvArgs a) {
  constexpr int BP = 16 * TP, BQ = 16 * TQ;
  constexpr int kRow = BP + 4;                          // LDS row of one q, padded
  __shared__ __attribute__((aligned(16))) float tile[BQ * kRow];   // the accumulators between waves, [q][p]
  __shared__ int64_t s_out[BQ];                         // output offset of each q; -1 past the end
  const ConvGeom g = a.g;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned id = (unsigned)gvv::xcd_contiguous(blockIdx.x, gridDim.x);
  const unsigned per_class = (unsigned)a.ptiles * (unsigned)a.qtiles;
  const int cls = (int)(id / per_class);
  const unsigned rest = id - (unsigned)cls * per_class;
  const int qt = (int)(rest / (unsigned)a.ptiles), pt = (int)(rest - (unsigned)qt * (unsigned)a.ptiles);
  const int ry = FWD ? 0 : cls / a.classes_x, rx = FWD ? 0 : cls - ry * a.classes_x;
  const Taps ty = axis_taps(FWD, g.KS, g.S, g.PAD, g.H, g.OH, ry), tx = axis_taps(FWD, g.KS, g.S, g.PAD, g.W, g.OW, rx);
  const int C = FWD ? g.Cin : g.Cout, P = FWD ? g.Cout : g.Cin;
  const int SH = FWD ? g.H : g.OH, SW = FWD ? g.W : g.OW;                     // source image
  const int DH = FWD ? g.OH : g.H, DW = FWD ? g.OW : g.W;                     // output image
  const int kstep = FWD ? 1 : g.S, dir = FWD ? 1 : -1, mul = FWD ? g.S : 1;
  const int64_t Q = int64_t(g.B) * ty.pixels * tx.pixels;
  const int64_t q0 = int64_t(qt) * BQ;
  if (q0 >= Q) return;                                  // smaller classes have fewer tiles
  const int p0 = pt * BP;
  const unsigned C8 = (unsigned)C >> 3;
  const unsigned chunks = (unsigned)(ty.n * tx.n) * C8;                       // 8-channel chunks of k
  const unsigned steps = (chunks + 3) / 4;
  const int row = lane & 15, kg = lane >> 4;

  // rows past P repeat the last one (their results are not stored); pixels past Q read nothing
  const uint16_t* wrow[TP];
#pragma unroll
  for (int i = 0; i < TP; ++i)
    wrow[i] = a.w + int64_t(min(p0 + 16 * i + row, P - 1)) * g.KS * g.KS * C + (ALIGNED ? 8 * kg : 0);
  const uint16_t* src[TQ];                              // source pixel (sy, sx), where tap (0, 0) reads
  int sy[TQ], sx[TQ];
  {
    const int per = ty.pixels * tx.pixels;
    const int64_t q = q0 + row;
    int b = quotient(q, per);
    const int r = int(q - int64_t(b) * per);
    int yc = r / tx.pixels, xc = r - yc * tx.pixels;
#pragma unroll
    for (int j = 0; j < TQ; ++j) {
      const bool live = q + 16 * j < Q;
      sy[j] = live ? yc * mul + ty.add : INT32_MIN / 2;
      sx[j] = xc * mul + tx.add;
      src[j] = a.src + ((int64_t(b) * SH + (live ? sy[j] : 0)) * SW + sx[j]) * C + (ALIGNED ? 8 * kg : 0);
      if (tid < 16)
        s_out[16 * j + row] = live ? ((int64_t(b) * DH + (FWD ? yc : yc * g.S + ry)) * DW + (FWD ? xc : xc * g.S + rx)) * P : -1;
      xc += 16;
      while (xc >= tx.pixels) {
        xc -= tx.pixels;
        if (++yc == ty.pixels) { yc = 0; ++b; }
      }
    }
  }

  f32x4 acc[TP][TQ];
#pragma unroll
  for (int i = 0; i < TP; ++i)
#pragma unroll
    for (int j = 0; j < TQ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  Words4 fa[NS][TP], fb[NS][TQ];
  // tap (t, u) and channel c of a chunk; ALIGNED: uniform over the wave
  auto load_tap = [&](int t, int u, unsigned c, bool live, Words4* va, Words4* vb) {
    const int64_t wofs = int64_t((ty.k0 + kstep * t) * g.KS + tx.k0 + kstep * u) * C + c;
    const int64_t sofs = (int64_t(dir * t) * SW + dir * u) * C + c;
#pragma unroll
    for (int i = 0; i < TP; ++i) {
      va[i] = Words4{{0, 0, 0, 0}};
      if (live) va[i] = *reinterpret_cast<const Words4*>(wrow[i] + wofs);
    }
#pragma unroll
    for (int j = 0; j < TQ; ++j) {
      vb[j] = Words4{{0, 0, 0, 0}};
      if (live && (unsigned)(sy[j] + dir * t) < (unsigned)SH && (unsigned)(sx[j] + dir * u) < (unsigned)SW)
        vb[j] = *reinterpret_cast<const Words4*>(src[j] + sofs);
    }
  };
  const unsigned len = min((unsigned)NS, (steps + NW - 1) / NW);    // of a stretch
  auto load_stretch = [&](unsigned first) {
    if (ALIGNED) {
      const unsigned per_tap = C8 / 4;
      unsigned tap = first / per_tap, c = first - tap * per_tap;
      int t = (int)(tap / (unsigned)max(tx.n, 1)), u = (int)tap - t * tx.n;
      t = __builtin_amdgcn_readfirstlane(t);
      u = __builtin_amdgcn_readfirstlane(u);
      c = __builtin_amdgcn_readfirstlane(c);
#pragma unroll
      for (int k = 0; k < NS; ++k)
        if (k < (int)len && first + k < steps) {
          load_tap(t, u, 32 * c, true, fa[k], fb[k]);
          if (++c == per_tap) {
            c = 0;
            if (++u == tx.n) { u = 0; ++t; }
          }
        }
    } else {
#pragma unroll
      for (int k = 0; k < NS; ++k)
        if (k < (int)len && first + k < steps) {
          const unsigned kc = (first + k) * 4 + kg;
          const unsigned tap = kc / C8, c = (kc - tap * C8) * 8;
          const int t = (int)(tap / (unsigned)tx.n), u = (int)tap - t * tx.n;
          load_tap(t, u, c, kc < chunks, fa[k], fb[k]);
        }
    }
  };
  float* mine = tile + row * kRow + 4 * kg;
  unsigned first = wave * len;                                      // this wave's stretch
  load_stretch(first);
  for (unsigned base = 0; base < steps; base += NW * len) {
    for (int turn = 0; turn < NW && base + turn * len < steps; ++turn) {
      if (turn == wave) {
        if (NW > 1 && first > 0) {
#pragma unroll
          for (int i = 0; i < TP; ++i)
#pragma unroll
            for (int j = 0; j < TQ; ++j) acc[i][j] = *reinterpret_cast<const f32x4*>(mine + 16 * j * kRow + 16 * i);
        }
#pragma unroll
        for (int k = 0; k < NS; ++k)
          if (k < (int)len && first + k < steps) {
#pragma unroll
            for (int i = 0; i < TP; ++i)
#pragma unroll
              for (int j = 0; j < TQ; ++j) acc[i][j] = mfma(as_bf16x8(fa[k][i]), as_bf16x8(fb[k][j]), acc[i][j]);
          }
        if (NW > 1) {
#pragma unroll
          for (int i = 0; i < TP; ++i)
#pragma unroll
            for (int j = 0; j < TQ; ++j) *reinterpret_cast<f32x4*>(mine + 16 * j * kRow + 16 * i) = acc[i][j];
        }
        first += NW * len;
        load_stretch(first);
      }
      if (NW > 1) __syncthreads();
    }
  }
  if (NW == 1 || steps == 0) {
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < TP; ++i)
#pragma unroll
        for (int j = 0; j < TQ; ++j) *reinterpret_cast<f32x4*>(mine + 16 * j * kRow + 16 * i) = acc[i][j];
    }
    __syncthreads();
  }

  // the epilogue: 8 consecutive p of one q per thread
  for (int e = tid; e < BQ * (BP / 8); e += 64 * NW) {
    const int ql = e / (BP / 8), pl = (e - ql * (BP / 8)) * 8;
    const int64_t so = s_out[ql];
    const int pb = p0 + pl;
    if (so < 0 || pb >= P) continue;                    // P is a multiple of 8
    float v[8];
    const float* t0 = tile + ql * kRow + pl;
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = t0[k];
    const int64_t o = so + pb;
    if (FWD) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        v[k] += a.bias[pb + k];
        if (a.relu) v[k] = v[k] > 0.f ? v[k] : 0.f;
      }
    } else if (a.mask) {
      uint16_t m[8];
      __builtin_memcpy(m, a.mask + o, 16);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (!(bf2f(m[k]) > 0.f)) v[k] = 0.f;
    }
    if (FWD && a.out_f32) {
      float* d = static_cast<float*>(a.out) + o;
      if (a.wide) {
        *reinterpret_cast<float4*>(d) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(d + 4) = make_float4(v[4], v[5], v[6], v[7]);
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) d[k] = v[k];
      }
      continue;
    }
    uint16_t* d = static_cast<uint16_t*>(a.out) + o;
    bf16x8 h;
#pragma unroll
    for (int k = 0; k < 8; ++k) h[k] = static_cast<__bf16>(v[k]);         // round to nearest even
    if (a.wide) *reinterpret_cast<bf16x8*>(d) = h;
    else __builtin_memcpy(d, &h, 16);
  }
}

// ---- backward weight -----------------------------------------------------------------------
// The reduction runs over pixels, which are strided in NHWC, while an MFMA operand wants 8
// consecutive k in a lane.  Each lane loads 8 pixels x 8 channels of x (8 pixels x NB channels of
// dz) with one vector load per pixel and transposes them in registers, one byte permute per pair
// of pixels and channel.  Fragment j then holds channel j of every lane's chunk: rows 8 r + j of
// the 128-row P tile (columns NB n + j of the 32-column Q tile, NB = 2), a fixed permutation that
// the epilogue undoes with 32-byte stores.  2-byte gathers into LDS took 385 us for the network's
// layers of 16 images, and the bias sums, formed here with a row of ones, 83 us of their own.
constexpr int kWP = 128, kWQ = 32;       // rows and columns of a tile; 128 x 64 halves the waves per SIMD: 131 us
                                         // against 111 for the network's seven layers at 16 images
constexpr int kWWaves = 4;               // waves of a workgroup, splitting its pixels
constexpr int64_t kWeightBlocks = 512, kWeightSteps = 4;   // weight_split

struct WeightArgs {
  ConvGeom g;
  const uint16_t* x;       // [B][H][W][Cin]
  const uint16_t* dz;      // [B][OH][OW][Cout]
  float* dw;               // splits > 1: partials [splits][Cout][P]; else the gradient itself
  float* db;               // [splits][Cout] or null
  int64_t per;             // pixels per split (a multiple of 32 kWWaves)
  int wide;                // dw is 16-byte aligned
};

__device__ __forceinline__ uint32_t lo_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t hi_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

__global__ __launch_bounds__(64 * kWWaves) void k_conv_weight(WeightArgs a) {
  constexpr int NB = kWQ / 16, kVals = 8 * NB * 4 + NB;   // per lane: 8 x NB fragments, and the bias column sums
  __shared__ float red[kWWaves / 2][kVals][64];
  const ConvGeom g = a.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 15, kg = lane >> 4;
  const int P = g.KS * g.KS * g.Cin, Q = g.Cout;
  const int64_t K = int64_t(g.B) * g.OH * g.OW;
  const int q0 = blockIdx.x * kWQ, p0 = blockIdx.y * kWP;
  const bool bias = a.db && blockIdx.y == 0;
  // this lane's chunk of 8 rows (one tap) and its NB columns; chunks past the end load nothing
  const int pc = p0 + 8 * row, qc = q0 + NB * row;
  const bool p_live = pc < P, q_live = qc < Q;
  const int tap = p_live ? pc / g.Cin : 0, ci = p_live ? pc - tap * g.Cin : 0;
  const int kh = tap / g.KS, kw = tap - kh * g.KS;
  const int64_t beg = int64_t(blockIdx.z) * a.per;
  const int64_t end = beg + a.per < K ? beg + a.per : K;

  uint32_t rx[8][4], rz[8][NB / 2];
  const int64_t xstep = int64_t(g.S) * g.Cin;
  const bool whole = g.OW % 8 == 0;          // a lane's 8 pixels lie in one row
  auto load = [&](int64_t k0) {
    int64_t k = k0 + 8 * kg;
    const int ohw = g.OH * g.OW;
    int b = quotient(k, ohw);
    const int r = int(k - int64_t(b) * ohw);
    int oh = r / g.OW, ow = r - oh * g.OW;
    const uint16_t* px = a.x + ((int64_t(b) * g.H + oh * g.S - g.PAD + kh) * g.W + ow * g.S - g.PAD + kw) * g.Cin + ci;
    const uint16_t* pz = a.dz + k * g.Cout + qc;
    const int live = int(end - k < 8 ? end - k : 8);        // pixels of this lane before the end
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int c = 0; c < 4; ++c) rx[i][c] = 0;
#pragma unroll
      for (int c = 0; c < NB / 2; ++c) rz[i][c] = 0;
      if (i < live) {
        const int ih = oh * g.S - g.PAD + kh, iw = ow * g.S - g.PAD + kw;
        if (p_live && (unsigned)ih < (unsigned)g.H && (unsigned)iw < (unsigned)g.W) __builtin_memcpy(rx[i], px, 16);
        if (q_live) __builtin_memcpy(rz[i], pz + i * int64_t(g.Cout), 2 * NB);
      }
      ++ow;
      px += xstep;
      if (!whole && ow == g.OW) {
        ow = 0;
        if (++oh == g.OH) { oh = 0; ++b; }
        px = a.x + ((int64_t(b) * g.H + oh * g.S - g.PAD + kh) * g.W - g.PAD + kw) * g.Cin + ci;
      }
    }
  };

  f32x4 acc[8][NB], accb[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    accb[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bf16x8 ones = as_bf16x8(Words4{{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u}});
  int64_t k0 = beg + 32 * wave;
  if (k0 < end) load(k0);
  for (; k0 < end; k0 += 32 * kWWaves) {
    bf16x8 fx[8], fz[NB];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      Words4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v.w[i] = c & 1 ? hi_halves(rx[2 * i][c / 2], rx[2 * i + 1][c / 2])
                                                 : lo_halves(rx[2 * i][c / 2], rx[2 * i + 1][c / 2]);
      fx[c] = as_bf16x8(v);
    }
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      Words4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v.w[i] = c & 1 ? hi_halves(rz[2 * i][c / 2], rz[2 * i + 1][c / 2])
                                                 : lo_halves(rz[2 * i][c / 2], rz[2 * i + 1][c / 2]);
      fz[c] = as_bf16x8(v);
    }
    if (k0 + 32 * kWWaves < end) load(k0 + 32 * kWWaves);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = mfma(fx[i], fz[j], acc[i][j]);
    if (bias) {
#pragma unroll
      for (int j = 0; j < NB; ++j) accb[j] = mfma(ones, fz[j], accb[j]);
    }
  }

  // sum the waves pairwise through LDS: (0 + 2), (1 + 3), then 0 + 1
#pragma unroll
  for (int half = kWWaves / 2; half >= 1; half >>= 1) {
    __syncthreads();
    if (wave >= half && wave < 2 * half) {
      float(*d)[64] = red[wave - half];
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) d[(i * NB + j) * 4 + r][lane] = acc[i][j][r];
#pragma unroll
      for (int j = 0; j < NB; ++j) d[32 * NB + j][lane] = accb[j][0];
    }
    __syncthreads();
    if (wave < half) {
      const float(*d)[64] = red[wave];
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] += d[(i * NB + j) * 4 + r][lane];
#pragma unroll
      for (int j = 0; j < NB; ++j) accb[j][0] += d[32 * NB + j][lane];
    }
  }
  if (wave != 0 || !q_live) return;
  // accumulator r of fragment pair (i, j): p = p0 + 8 (4 kg + r) + i, q = q0 + NB row + j
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int q = qc + j;
    if (q >= Q) continue;
    if (bias && kg == 0) a.db[int64_t(blockIdx.z) * Q + q] = accb[j][0];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int p = p0 + 8 * (4 * kg + r);
      if (p >= P) continue;
      float* o = a.dw + (int64_t(blockIdx.z) * Q + q) * P + p;
      if (a.wide) {
        *reinterpret_cast<float4*>(o) = make_float4(acc[0][j][r], acc[1][j][r], acc[2][j][r], acc[3][j][r]);
        *reinterpret_cast<float4*>(o + 4) = make_float4(acc[4][j][r], acc[5][j][r], acc[6][j][r], acc[7][j][r]);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = acc[i][j][r];
      }
    }
  }
}

// dw[i] = sum_s part[s][i] and db likewise, deterministic.  Block: 64 consecutive outputs x 16
// split lanes; each lane sums every 16th split, then the 16 partial sums are added in order.
constexpr int kSumLanes = 16;
__global__ __launch_bounds__(64 * kSumLanes) void k_split_sum(const float* __restrict__ part, const float* __restrict__ bpart,
                                                              int splits, int64_t n, int nb, float* __restrict__ out,
                                                              float* __restrict__ bout) {
  __shared__ float red[kSumLanes][64];
  const int64_t wblocks = (n + 63) / 64;
  const bool is_bias = (int64_t)blockIdx.x >= wblocks;
  const float* src = is_bias ? bpart : part;
  float* dst = is_bias ? bout : out;
  const int64_t m = is_bias ? nb : n;
  const int64_t i = (int64_t(blockIdx.x) - (is_bias ? wblocks : 0)) * 64 + (threadIdx.x & 63);
  const int r = threadIdx.x >> 6;
  float s = 0.f;
  if (i < m) {
#pragma unroll 4
    for (int k = r; k < splits; k += kSumLanes) s += src[int64_t(k) * m + i];
  }
  red[r][threadIdx.x & 63] = s;
  __syncthreads();
  if (r == 0 && i < m) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < kSumLanes; ++k) t += red[k][threadIdx.x];
    dst[i] = t;
  }
}

// fp32 master weights [Cout][T][Cin] -> bf16 copy and bf16 transpose [Cin][T][Cout], for up to
// kPrepareLayers layers in one launch (a launch of its own per layer took 4 us each, 5 to 7 layers
// of them idle): layer l owns blocks [start[l], start[l + 1]).
// Bound by memory (8 bytes a weight; 1.65 M weights 2.6 us at the copy rate) and latency.  A block
// takes kPrepCo rows x kPrepJ columns of the layer as a matrix [Cout][T * Cin] and turns them in LDS,
// so that loads and both stores are runs of 64 bytes and more: one thread per weight with its
// transposed store 2 bytes wide, each to a line of its own, took 13.8 us, this 8.4.
constexpr int kPrepareLayers = 16, kPrepCo = 32, kPrepJ = 64;
struct PrepareArgs {
  const float* w[kPrepareLayers];
  uint16_t* wb[kPrepareLayers];
  uint16_t* wt[kPrepareLayers];
  int cout[kPrepareLayers], taps[kPrepareLayers], cin[kPrepareLayers];
  unsigned start[kPrepareLayers + 1];
  int n;
};

__global__ __launch_bounds__(256) void k_prepare_weights(PrepareArgs a) {
  __shared__ uint16_t tile[kPrepJ][kPrepCo + 2];         // rows 17 words apart: no two lanes of a store share a bank
  int l = 0;
  while (l + 1 < a.n && blockIdx.x >= a.start[l + 1]) ++l;
  const int Cout = a.cout[l], T = a.taps[l], Cin = a.cin[l];
  const int64_t row = int64_t(T) * Cin;
  const unsigned jblocks = unsigned((row + kPrepJ - 1) / kPrepJ), blk = blockIdx.x - a.start[l];
  const int co0 = int(blk / jblocks) * kPrepCo;
  const int64_t j0 = int64_t(blk % jblocks) * kPrepJ;
  {
    const int dj = threadIdx.x % kPrepJ, r = threadIdx.x / kPrepJ;
    constexpr int kRows = 256 / kPrepJ, kLoads = kPrepCo / kRows;
    float v[kLoads];
#pragma unroll
    for (int k = 0; k < kLoads; ++k) {
      const int co = co0 + r + kRows * k;
      v[k] = co < Cout && j0 + dj < row ? a.w[l][co * row + j0 + dj] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < kLoads; ++k) {
      const int co = co0 + r + kRows * k;
      const uint16_t h = f2bf(v[k]);
      if (co < Cout && j0 + dj < row) a.wb[l][co * row + j0 + dj] = h;
      tile[dj][co - co0] = h;
    }
  }
  if (!a.wt[l]) return;
  __syncthreads();
  const int co = co0 + int(threadIdx.x % kPrepCo);
  if (co >= Cout) return;
  const int64_t t0 = j0 / Cin;
  for (int dj = threadIdx.x / kPrepCo; dj < kPrepJ && j0 + dj < row; dj += 256 / kPrepCo) {
    int64_t ci = j0 - t0 * Cin + dj, t = t0;              // column of the matrix: tap and input channel
    while (ci >= Cin) ci -= Cin, ++t;
    a.wt[l][(ci * T + t) * Cout + co] = tile[dj][co - co0];
  }
}

// Renders [B][V][h][w][3] fp32 -> NHWC8 bf16 mosaic [B][rows*h/d][cols*w/d][8]: view v at tile
// (v / cols, v % cols), each output pixel the mean of a d x d block.  features == 0: channels
// 0..2 RGB, 3..7 zero.  features == 1: channels 0..2 RGB - 0.5, 3 the covered fraction of the
// block (pixels other than the (0, 1, 0) background), 4..5 the tile-local x and y in [-1, 1],
// 6..7 zero.  Empty tiles are zero.
__global__ void k_pack_mosaic(const float* __restrict__ render, int B, int V, int h, int w, int cols, int d,
                              int features, uint16_t* __restrict__ x) {
  const int rows = (V + cols - 1) / cols;
  const int th = h / d, tw = w / d;
  const int H = rows * th, W = cols * tw;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= int64_t(B) * H * W) return;
  const int X = int(i % W);
  const int64_t r = i / W;
  const int Y = int(r % H), b = int(r / H);
  const int v = (Y / th) * cols + X / tw;
  uint16_t c[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (v < V) {
    float acc[3] = {0.f, 0.f, 0.f};
    int covered = 0;
    const int y0 = (Y % th) * d, x0 = (X % tw) * d;
    for (int yy = 0; yy < d; ++yy) {
      const float* s = render + ((((int64_t(b) * V + v) * h) + y0 + yy) * w + x0) * 3;
      for (int xx = 0; xx < d; ++xx) {
        const float R = s[3 * xx], G = s[3 * xx + 1], Bc = s[3 * xx + 2];
        acc[0] += R;
        acc[1] += G;
        acc[2] += Bc;
        covered += !(R == 0.f && G == 1.f && Bc == 0.f);
      }
    }
    const float inv = 1.f / float(d * d);
    const float off = features ? 0.5f : 0.f;
    c[0] = f2bf(acc[0] * inv - off); c[1] = f2bf(acc[1] * inv - off); c[2] = f2bf(acc[2] * inv - off);
    if (features) {
      c[3] = f2bf(covered * inv);
      c[4] = f2bf(2.f * ((X % tw) + 0.5f) / float(tw) - 1.f);
      c[5] = f2bf(2.f * ((Y % th) + 0.5f) / float(th) - 1.f);
    }
  }
  *reinterpret_cast<uint4*>(x + i * 8) = make_uint4(c[0] | (uint32_t(c[1]) << 16), c[2] | (uint32_t(c[3]) << 16),
                                                    c[4] | (uint32_t(c[5]) << 16), 0);
}

bool geom_ok(const ConvGeom& g, std::string& why) {
  if (g.B <= 0 || g.H <= 0 || g.W <= 0 || g.Cin <= 0 || g.Cout <= 0 || g.KS <= 0 || g.S <= 0 || g.PAD < 0) {
    why = "conv: sizes must be positive (pad >= 0)";
    return false;
  }
  if (g.Cin % 8 || g.Cout % 8) {
    why = "conv: channel counts must be multiples of 8 (NHWC8 layout), got Cin=" + std::to_string(g.Cin) +
          " Cout=" + std::to_string(g.Cout);
    return false;
  }
  if (g.OH <= 0 || g.OW <= 0) {
    why = "conv: kernel larger than the padded input";
    return false;
  }
  if (int64_t(g.B) * g.H * g.W * g.Cin >= (int64_t(1) << 40)) {
    why = "conv: input too large";
    return false;
  }
  return true;
}

ConvGeom make_geom(int B, int H, int W, int Cin, int Cout, int ks, int stride, int pad) {
  ConvGeom g{B, H, W, Cin, 0, 0, Cout, ks, stride, pad};
  if (stride > 0) {
    g.OH = (H + 2 * pad - ks) / stride + 1;
    g.OW = (W + 2 * pad - ks) / stride + 1;
  }
  return g;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int hip_status(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gvv::set_last_error(std::string(what) + ": " + hipGetErrorString(e));
  return 0;
}

template <bool FWD, int TP, int TQ, int NW, int NS>
int launch(ConvArgs a, hipStream_t s, const char* what) {
  const ConvGeom& g = a.g;
  const int cy = FWD ? 1 : (g.S < g.H ? g.S : g.H), cx = FWD ? 1 : (g.S < g.W ? g.S : g.W);
  // the class of residue 0 has the most pixels
  const int64_t Q = FWD ? int64_t(g.B) * g.OH * g.OW
                        : int64_t(g.B) * ((g.H + g.S - 1) / g.S) * ((g.W + g.S - 1) / g.S);
  const int P = FWD ? g.Cout : g.Cin;
  a.ptiles = (P + 16 * TP - 1) / (16 * TP);
  const int64_t qtiles = (Q + 16 * TQ - 1) / (16 * TQ);
  const int64_t blocks = qtiles * a.ptiles * cy * cx;
  if (blocks > INT32_MAX) return gvv::set_last_error(std::string(what) + ": too many output tiles");
  a.qtiles = int(qtiles);
  a.classes_x = cx;
  if ((FWD ? g.Cin : g.Cout) % 32 == 0)
    hipLaunchKernelGGL((k_conv<FWD, true, TP, TQ, NW, NS>), dim3(unsigned(blocks)), dim3(64 * NW), 0, s, a);
  else
    hipLaunchKernelGGL((k_conv<FWD, false, TP, TQ, NW, NS>), dim3(unsigned(blocks)), dim3(64 * NW), 0, s, a);
  return hip_status(what);
}

// Tile choice: the largest tile that still gives the chip's 1024 SIMDs a wave each, as a larger
// tile reads its operands fewer times, or failing that its 256 CUs a workgroup each.  With 1024 tiles
// and more, one wave per tile fills the chip and passes no accumulators (backward data of the
// 64-channel layer at 16 images: 29 us against 38 with four waves, of the 128-channel layer 24 against
// 28); 64 x 128 tiles, where there are so many, take 58 us against 70 with 64 x 64 (128 -> 128 channels,
// 3 x 3, stride 1, 4 x 128^2; staged through LDS 65) and 105 against 134 (256 -> 256, 8 x 64^2; 146), but
// 44 against 41 over a reduction of 9 steps (32 -> 64, stride 2, 64 x 128^2), where the output counts.  With
// fewer, the stretches of the reduction are loaded side by side: 64 x 64 tiles by two waves, as with four
// the accumulators travel twice as far (64 -> 64, 3 x 3, stride 1, 16 x 56^2: 21 us, 28 with four waves,
// staged through LDS 22; the 64 -> 128 layer of 16 images 14.4 against 15.4); smaller tiles all at once where the waves' registers hold them (the 4096-deep
// head of one image: 13 us with 16 waves, 21 with 8 and two rounds of loads, 75 with one wave; the
// 2304-deep layer 9.4 us with 8 waves, 11.8 with 16, whose accumulators travel twice as far).
template <bool FWD>
int launch_conv(const ConvArgs& a, hipStream_t s, const char* what) {
  const ConvGeom& g = a.g;
  const int64_t Q = FWD ? int64_t(g.B) * g.OH * g.OW : int64_t(g.B) * g.H * g.W;
  const int64_t P = FWD ? g.Cout : g.Cin;
  const int taps = FWD ? g.KS : (g.KS + g.S - 1) / g.S;            // of one axis, at most
  const int64_t steps = (int64_t(taps) * taps * (FWD ? g.Cin : g.Cout) + 31) / 32;
  auto tiles = [&](int bp, int bq) { return ((P + bp - 1) / bp) * ((Q + bq - 1) / bq); };
  if (P <= 32 && tiles(32, 64) >= 1024) return launch<FWD, 2, 4, 1, 2>(a, s, what);
  if (P <= 32 && tiles(32, 64) >= 256) return launch<FWD, 2, 4, 4, 3>(a, s, what);
  if (P > 32 && steps >= 16 && tiles(64, 128) >= 1024) return launch<FWD, 4, 8, 1, 2>(a, s, what);
  if (P > 32 && tiles(64, 64) >= 1024) return launch<FWD, 4, 4, 1, 2>(a, s, what);
  if (P > 32 && tiles(64, 64) >= 256) return launch<FWD, 4, 4, 2, 3>(a, s, what);
  if (P > 16 && tiles(32, 32) >= 256) return launch<FWD, 2, 2, 8, 5>(a, s, what);
  if (steps < 16) return launch<FWD, 1, 1, 4, 4>(a, s, what);
  return steps <= 80 ? launch<FWD, 1, 1, 8, 10>(a, s, what) : launch<FWD, 1, 1, 16, 8>(a, s, what);
}

// Split of the weight-gradient reduction over workgroups: enough workgroups for the chip
// (about 512 of four waves), each with at least 4 steps of 32 pixels per wave, which keeps the
// partial sums (read once more by k_split_sum) a small share of the traffic.
void weight_split(const ConvGeom& g, int& splits, int64_t& per) {
  const int64_t P = int64_t(g.KS) * g.KS * g.Cin, K = int64_t(g.B) * g.OH * g.OW;
  const int64_t tiles = ((P + kWP - 1) / kWP) * ((g.Cout + kWQ - 1) / kWQ);
  constexpr int64_t unit = 32 * kWWaves;               // pixels of one step of every wave
  const int64_t steps = (K + unit - 1) / unit;
  int64_t want = (kWeightBlocks + tiles - 1) / tiles;
  if (want > steps / kWeightSteps) want = steps / kWeightSteps;
  if (want < 1) want = 1;
  per = ((steps + want - 1) / want) * unit;
  splits = int((K + per - 1) / per);
}

}  // namespace

extern "C" {

int gvv_conv_out_size(int32_t in, int32_t ks, int32_t stride, int32_t pad) {
  if (stride <= 0) return 0;
  return (in + 2 * pad - ks) / stride + 1;
}

int gvv_conv_forward(int32_t B, int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t ks, int32_t stride,
                     int32_t pad, const void* x, const void* w, const float* bias, int32_t relu, void* y,
                     int32_t y_f32, void* stream) {
  const ConvGeom g = make_geom(B, H, W, Cin, Cout, ks, stride, pad);
  std::string why;
  if (!geom_ok(g, why)) return gvv::set_last_error(why);
  if (!x || !w || !bias || !y) return gvv::set_last_error("conv forward: null pointer");
  if (!aligned16(x) || !aligned16(w)) return gvv::set_last_error("conv forward: x and w must be 16-byte aligned");
  ConvArgs a{};
  a.g = g;
  a.src = static_cast<const uint16_t*>(x);
  a.w = static_cast<const uint16_t*>(w);
  a.bias = bias;
  a.out = y;
  a.out_f32 = y_f32 ? 1 : 0;
  a.relu = relu ? 1 : 0;
  a.wide = aligned16(y) ? 1 : 0;
  return launch_conv<true>(a, static_cast<hipStream_t>(stream), "conv forward");
}

int gvv_conv_backward_data(int32_t B, int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t ks, int32_t stride,
                           int32_t pad, const void* dz, const void* wt, const void* x_mask, void* dx, void* stream) {
  const ConvGeom g = make_geom(B, H, W, Cin, Cout, ks, stride, pad);
  std::string why;
  if (!geom_ok(g, why)) return gvv::set_last_error(why);
  if (!dz || !wt || !dx) return gvv::set_last_error("conv backward data: null pointer");
  if (!aligned16(dz) || !aligned16(wt)) return gvv::set_last_error("conv backward data: dz and wt must be 16-byte aligned");
  ConvArgs a{};
  a.g = g;
  a.src = static_cast<const uint16_t*>(dz);
  a.w = static_cast<const uint16_t*>(wt);
  a.mask = static_cast<const uint16_t*>(x_mask);
  a.out = dx;
  a.wide = aligned16(dx) ? 1 : 0;
  return launch_conv<false>(a, static_cast<hipStream_t>(stream), "conv backward data");
}

int64_t gvv_conv_workspace_floats(int32_t B, int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t ks,
                                  int32_t stride, int32_t pad) {
  const ConvGeom g = make_geom(B, H, W, Cin, Cout, ks, stride, pad);
  std::string why;
  if (!geom_ok(g, why)) return -1;
  int splits;
  int64_t per;
  weight_split(g, splits, per);
  return int64_t(splits) * Cout * ks * ks * Cin + int64_t(splits) * Cout;
}

int gvv_conv_backward_weight(int32_t B, int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t ks, int32_t stride,
                             int32_t pad, const void* x, const void* dz, float* dw, float* db, float* workspace,
                             int64_t workspace_floats, void* stream) {
  const ConvGeom g = make_geom(B, H, W, Cin, Cout, ks, stride, pad);
  std::string why;
  if (!geom_ok(g, why)) return gvv::set_last_error(why);
  if (!x || !dz || !dw || !workspace) return gvv::set_last_error("conv backward weight: null pointer");
  const int64_t need = gvv_conv_workspace_floats(B, H, W, Cin, Cout, ks, stride, pad);
  if (workspace_floats < need)
    return gvv::set_last_error("conv backward weight: workspace holds " + std::to_string(workspace_floats) +
                               " floats, needs " + std::to_string(need));
  hipStream_t s = static_cast<hipStream_t>(stream);
  int splits;
  int64_t per;
  weight_split(g, splits, per);
  const int64_t P = int64_t(ks) * ks * Cin, n = P * Cout;
  const int64_t ptiles = (P + kWP - 1) / kWP;
  if (P > INT32_MAX - kWP || ptiles > 65535 || splits > 65535)
    return gvv::set_last_error("conv backward weight: too many weight rows");
  WeightArgs a{};
  a.g = g;
  a.x = static_cast<const uint16_t*>(x);
  a.dz = static_cast<const uint16_t*>(dz);
  a.dw = splits > 1 ? workspace : dw;
  a.db = !db ? nullptr : splits > 1 ? workspace + int64_t(splits) * n : db;
  a.per = per;
  a.wide = aligned16(a.dw) ? 1 : 0;
  const dim3 grid(unsigned((Cout + kWQ - 1) / kWQ), unsigned(ptiles), unsigned(splits));
  hipLaunchKernelGGL(k_conv_weight, grid, dim3(64 * kWWaves), 0, s, a);
  if (splits > 1) {
    const unsigned blocks = unsigned((n + 63) / 64 + (db ? (Cout + 63) / 64 : 0));
    hipLaunchKernelGGL(k_split_sum, dim3(blocks), dim3(64 * kSumLanes), 0, s, workspace, a.db, splits, n, Cout, dw, db);
  }
  return hip_status("conv backward weight");
}

int gvv_conv_prepare_weights_layers(int32_t n, const int32_t* Cout, const int32_t* taps, const int32_t* Cin,
                                    const float* const* w, void* const* w_bf16, void* const* wt_bf16, void* stream) {
  if (n <= 0 || !Cout || !taps || !Cin || !w || !w_bf16 || !wt_bf16)
    return gvv::set_last_error("prepare weights: need at least one layer and its tables");
  for (int32_t l = 0; l < n; ++l) {
    if (Cout[l] <= 0 || taps[l] <= 0 || Cin[l] <= 0) return gvv::set_last_error("prepare weights: sizes must be positive");
    if (!w[l] || !w_bf16[l]) return gvv::set_last_error("prepare weights: null pointer");
  }
  for (int32_t l0 = 0; l0 < n; l0 += kPrepareLayers) {
    PrepareArgs a{};
    int64_t blocks = 0;
    for (int32_t l = l0; l < n && l < l0 + kPrepareLayers; ++l) {
      const int k = l - l0;
      a.w[k] = w[l];
      a.wb[k] = static_cast<uint16_t*>(w_bf16[l]);
      a.wt[k] = static_cast<uint16_t*>(wt_bf16[l]);
      a.cout[k] = Cout[l]; a.taps[k] = taps[l]; a.cin[k] = Cin[l];
      a.start[k] = unsigned(blocks);
      blocks += ((int64_t(Cout[l]) + kPrepCo - 1) / kPrepCo) * ((int64_t(taps[l]) * Cin[l] + kPrepJ - 1) / kPrepJ);
      if (blocks > INT32_MAX) return gvv::set_last_error("prepare weights: too many weights");
      a.n = k + 1;
      a.start[k + 1] = unsigned(blocks);
    }
    hipLaunchKernelGGL(k_prepare_weights, dim3(unsigned(blocks)), dim3(256), 0, static_cast<hipStream_t>(stream), a);
  }
  return hip_status("prepare weights");
}

int gvv_conv_prepare_weights(int32_t Cout, int32_t taps, int32_t Cin, const float* w, void* w_bf16, void* wt_bf16,
                             void* stream) {
  return gvv_conv_prepare_weights_layers(1, &Cout, &taps, &Cin, &w, &w_bf16, &wt_bf16, stream);
}

int gvv_pack_mosaic(const float* render, int32_t B, int32_t V, int32_t h, int32_t w, int32_t cols, int32_t down,
                    int32_t features, void* x, void* stream) {
  if (B <= 0 || V <= 0 || h <= 0 || w <= 0 || cols <= 0 || down <= 0)
    return gvv::set_last_error("pack mosaic: sizes must be positive");
  if (h % down || w % down) return gvv::set_last_error("pack mosaic: view size must be a multiple of the downsampling");
  if (features != 0 && features != 1) return gvv::set_last_error("pack mosaic: features must be 0 or 1");
  if (!render || !x || !aligned16(x)) return gvv::set_last_error("pack mosaic: null or misaligned pointer");
  const int rows = (V + cols - 1) / cols;
  const int64_t n = int64_t(B) * rows * (h / down) * cols * (w / down);
  hipLaunchKernelGGL(k_pack_mosaic, dim3(unsigned((n + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     render, B, V, h, w, cols, down, features, static_cast<uint16_t*>(x));
  return hip_status("pack mosaic");
}

}  // extern "C"
