// fs_unet.hip -- the learned proposal's network: a 4-level convolutional
// U-Net in BF16 on the MFMA units (v_mfma_f32_16x16x32_bf16, FP32
// accumulation) with hand-written forward and backward kernels and Adam on
// FP32 master weights.  No reference counterpart: the network ranks candidate
// (K, U, m) parameter sets for an inverse problem so that only the best few
// go to the exact time-step.
//
// Network (input H x W, H and W multiples of 32):
//   input  8 channels: initial terrain, 3 parameter channels, 4 zero
//   enc L  conv3x3+ReLU, conv3x3+ReLU at widths 32, 64, 128, 160 for levels
//          0..3, 2x2 average pooling between levels
//   dec L  nearest 2x upsampling of level L+1, concatenated with level L's
//          encoder output, then conv3x3+ReLU twice (widths 128, 64, 32)
//   head   1x1 conv to one channel (FP32)
// Activations are NHWC BF16; weights are FP32 masters with two BF16 copies:
// [tap][out][in] for the forward conv and [flipped tap][in][out] for the
// data gradient, which is then the same implicit GEMM.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "fs_conv_rows.h"
#include "fs_internal.h"
#include "fs_hostutil.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kInChannels = FS_UNET_IN_CHANNELS;
constexpr int kLevels = 4;
constexpr int kWidth[kLevels] = {32, 64, 128, 160};

__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);   // round to nearest even
  return static_cast<uint16_t>(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) {
  return __uint_as_float(static_cast<uint32_t>(h) << 16);
}

__device__ __forceinline__ f32x4 mfma16(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// 3x3 convolution, stride 1, zero padding, as an implicit GEMM:
//   out[p][n] = bias[n] + sum_{t, c} in[p + off_t][c] * wt[t][n][c]
// A wave computes 16 columns x R rows x 32 outputs of one image on
// v_mfma_f32_16x16x32_bf16: operand A the weights (row = output), operand B
// the pixels (column = pixel lane%16, 8 channels per lane group lane/16), so a
// lane ends with 8 consecutive outputs of one pixel (one 16-byte store).
//
// Per step of 32 input channels the wave holds its 9 taps' weights in
// registers and walks down the R + 2 input rows: a row is loaded once (16
// bytes per lane, straight from memory: no staging), its two column shifts
// are lane shifts within the 16 lanes of a row (DPP; the edge pixel comes from
// a second load that only lanes 0 and 15 take), and it feeds three output
// rows.  That is 9 * 2 * R MFMAs for R + 2 row loads and 18 weight reads; the
// kernel it replaces read two operands from LDS per MFMA pair and was bound by
// LDS (9 * 6 reads for 72 MFMAs per wave).  Row p of the next step (or of the
// wave's next tile) is requested as soon as row p of this one is used.
//
// The upsampled and concatenated decoder inputs are read where they lie, and
// the pooling, the ReLU gradient and the gradient of the upsampling happen on
// the finished tile, so none of them is a pass over memory of its own.
// Ranking 256 candidates at 256 x 256: 12.75 -> 7.43 ms (391 -> 672 TFLOP/s);
// the widest layers run at 820 to 990 TFLOP/s, the 32-channel layers of the
// top level at 3.4 TB/s.  Over all layers of a training step the matrix units are
// busy 27% of the cycles, LDS 8%, and waves wait 46% of theirs: two share a SIMD
// (253 registers), and the latency of their rows bounds them.
//
// Each accumulator adds its taps in order 0..8 within a step and the
// steps in order, so the sums are those of a plain loop over (channel step,
// tap), bit for bit, at every R.  kTapOuter (levels smaller than 8 x 16): those
// of the loop over (tap, channel step), the order these levels have always been
// summed in; their outputs keep their bits.
// ---------------------------------------------------------------------------
constexpr int kNB = 32;            // outputs per wave
constexpr int kKC = 32;            // input channels per step
constexpr int kWaves = 4;          // waves per workgroup
constexpr int kWFrags = 9 * (kNB / 16);
constexpr int kRsrc = 0x00020000;  // raw (unformatted) buffer, gfx9
constexpr uint32_t kOob = 0x80000000u;   // beyond every row: loads give zero

// The input: channels [0, ca) from a -- at half the resolution when up (a 2x
// nearest upsampling) -- and then cb channels from b.
struct ConvSrc {
  const uint16_t *a, *b;
  int ca, cb, up;
};
// The output.  Outputs [0, c1) (c1 = 0 but for the gradient of a
// concatenation) are summed over 2 x 2 pixels into lo, the others go to out;
// mask / lo_mask: zero where that tensor is not positive (ReLU gradient);
// pool: also the 2 x 2 averages of out.
struct ConvDst {
  uint16_t *out, *pool, *lo;
  const uint16_t *mask, *lo_mask;
  int c1;
};

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u32x4 load_px(const char *row, int bytes, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(row), 0, bytes, kRsrc),
      static_cast<int>(off), 0, 0);
}
// off: the lane's offset in bytes bytes, base: the wave's on top of it
__device__ __forceinline__ u32x4 load_px_at(const char *p, int bytes, uint32_t off, int base) {
  return __builtin_amdgcn_raw_buffer_load_b128(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(p), 0, bytes, kRsrc),
      static_cast<int>(off), base, 0);
}
// lane r's value from lane r-1 / r+1 of its 16; lanes 0 / 15 take edge's own
__device__ __forceinline__ u32x4 from_left(u32x4 v, u32x4 edge) {
  u32x4 o;
#pragma unroll
  for (int k = 0; k < 4; k++)
    o[k] = __builtin_amdgcn_update_dpp(edge[k], v[k], 0x111, 0xF, 0xF, false);
  return o;
}
__device__ __forceinline__ u32x4 from_right(u32x4 v, u32x4 edge) {
  u32x4 o;
#pragma unroll
  for (int k = 0; k < 4; k++)
    o[k] = __builtin_amdgcn_update_dpp(edge[k], v[k], 0x101, 0xF, 0xF, false);
  return o;
}
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// two floats to bf16 (round to nearest even), low half first
__device__ __forceinline__ uint32_t pack_bf(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}
// halves of g where the same half of y is positive, zero elsewhere
__device__ __forceinline__ uint32_t relu_mask(uint32_t g, uint32_t y) {
  const uint32_t lo = y & 0xFFFFu, hi = y >> 16;
  return ((lo != 0 && lo < 0x8000u) ? (g & 0xFFFFu) : 0u) |
         ((hi != 0 && hi < 0x8000u) ? (g & 0xFFFF0000u) : 0u);
}
__device__ __forceinline__ float bf_lo(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf_hi(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }
// sum of a 2 x 2 pixel block (this lane and the next, two rows), in the order
// (0,0), (0,1), (1,0), (1,1), times scale; right in the even lanes
__device__ __forceinline__ u32x4 block2x2(u32x4 r0, u32x4 r1, float scale) {
  u32x4 o;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t n0 = __builtin_amdgcn_mov_dpp(r0[k], 0xB1, 0xF, 0xF, true);
    const uint32_t n1 = __builtin_amdgcn_mov_dpp(r1[k], 0xB1, 0xF, 0xF, true);
    const float l = 0.f + bf_lo(r0[k]) + bf_lo(n0) + bf_lo(r1[k]) + bf_lo(n1);
    const float h = 0.f + bf_hi(r0[k]) + bf_hi(n0) + bf_hi(r1[k]) + bf_hi(n1);
    o[k] = pack_bf(scale * l, scale * h);
  }
  return o;
}

// Position of a wave's tile: image, first row and column.
struct TileAt {
  long b;
  int y0, x0;
  bool valid;
};
template <int R>
__device__ __forceinline__ TileAt tile_at(int tile, int ntiles, int tiles_x, int tiles_y) {
  TileAt t;
  t.valid = tile < ntiles;
  const int q = t.valid ? tile : 0;
  const int row = q / tiles_x;
  t.x0 = (q - row * tiles_x) * 16;
  t.b = row / tiles_y;
  t.y0 = (row % tiles_y) * R;
  return t;
}

// Bias, ReLU, rounding and the stores of a finished tile: acc[y][nt][i] is
// output n0 + 8 * (lane / 16) + 4 * nt + i of pixel (t.y0 + y, t.x0 + lane % 16).
template <int R>
__device__ __forceinline__ void store_tile(const f32x4 (&acc)[R][2], const TileAt &t,
                                           const ConvDst &dst, const float *bias, int relu,
                                           int n0, int nout, int H, int W) {
  if (!t.valid) return;
  const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  float bb[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (bias) {
#pragma unroll
    for (int k = 0; k < 8; k++) bb[k] = bias[n0 + 8 * g + k];
  }
  const bool to_lo = n0 < dst.c1;                 // uniform
  const int C = nout - dst.c1, n = n0 - dst.c1 + 8 * g;
  const int xx = t.x0 + r;
#pragma unroll
  for (int y = 0; y < R; y += 2) {
    u32x4 v[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      float f[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        f[k] = acc[y + h][k >> 2][k & 3] + bb[k];
        if (relu) f[k] = fmaxf(f[k], 0.f);
      }
#pragma unroll
      for (int k = 0; k < 4; k++) v[h][k] = pack_bf(f[2 * k], f[2 * k + 1]);
    }
    if (t.y0 + y >= H) break;                     // H is even
    const long px = (t.b * H + t.y0 + y) * W + xx;
    const long half = ((t.b * (H >> 1)) + ((t.y0 + y) >> 1)) * (W >> 1) + (xx >> 1);
    if (to_lo) {
      u32x4 s = block2x2(v[0], v[1], 1.f);
      if (xx < W && (r & 1) == 0) {
        const long at = half * dst.c1 + n0 + 8 * g;
        if (dst.lo_mask) {
          const u32x4 m = *reinterpret_cast<const u32x4 *>(dst.lo_mask + at);
#pragma unroll
          for (int k = 0; k < 4; k++) s[k] = relu_mask(s[k], m[k]);
        }
        *reinterpret_cast<u32x4 *>(dst.lo + at) = s;
      }
      continue;
    }
    if (dst.pool) {
      const u32x4 s = block2x2(v[0], v[1], 0.25f);
      if (xx < W && (r & 1) == 0) *reinterpret_cast<u32x4 *>(dst.pool + half * C + n) = s;
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (xx >= W) continue;
      const long at = (px + static_cast<long>(h) * W) * C + n;
      if (dst.mask) {
        const u32x4 m = *reinterpret_cast<const u32x4 *>(dst.mask + at);
#pragma unroll
        for (int k = 0; k < 4; k++) v[h][k] = relu_mask(v[h][k], m[k]);
      }
      *reinterpret_cast<u32x4 *>(dst.out + at) = v[h];
    }
  }
}

// output of MFMA row m in weight tile nt (see store_tile)
__device__ __forceinline__ int frag_out(int m, int nt) { return 8 * (m >> 2) + 4 * nt + (m & 3); }

// A workgroup keeps one block of 32 outputs and takes groups of kWaves tiles
// in turn; each XCD gets one contiguous run of groups (tiles that share input
// rows share an L2) for every block of outputs.  gridDim.x is a multiple of
// 8 * nout / 32.
template <int R>
__global__ __launch_bounds__(64 * kWaves, 2) void k_conv(ConvSrc src,
                                                         const uint16_t *__restrict__ wt,
                                                         const float *__restrict__ bias, int relu,
                                                         ConvDst dst, int nout, int H, int W,
                                                         int tiles_x, int tiles_y, int ntiles,
                                                         int groups) {
  // the step's weights in fragment order: [buffer][frag][lane]
  __shared__ u32x4 ws[2][kWFrags * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int nblk = nout / kNB;
  const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
  const int n0 = (q % nblk) * kNB, per = gridDim.x / (8 * nblk);
  const int g1 = static_cast<int>(static_cast<long>(groups) * (xcd + 1) / 8);
  const int first = static_cast<int>(static_cast<long>(groups) * xcd / 8) + q / nblk;
  if (first >= g1) return;
  const int cin = src.ca + src.cb;
  const int csteps = (cin + kKC - 1) / kKC;

  // ---- weights: global -> registers -> LDS, one step ahead ----
  constexpr int kWVec = 9 * kNB * 4;               // 16-byte vectors per step
  constexpr int kWPer = (kWVec + 64 * kWaves - 1) / (64 * kWaves);
  u32x4 wreg[kWPer];
  auto fetch_weights = [&](int c0) {
#pragma unroll
    for (int k = 0; k < kWPer; k++) {
      const int v = k * 64 * kWaves + static_cast<int>(threadIdx.x);
      const int row = v >> 2, c = c0 + 8 * (v & 3);
      const int t = row / kNB, o = row % kNB;
      wreg[k] = u32x4{0u, 0u, 0u, 0u};
      if (v < kWVec && c < cin)
        wreg[k] = *reinterpret_cast<const u32x4 *>(
            wt + (static_cast<long>(t) * nout + n0 + o) * cin + c);
    }
  };
  auto stage_weights = [&](int buf) {
#pragma unroll
    for (int k = 0; k < kWPer; k++) {
      const int v = k * 64 * kWaves + static_cast<int>(threadIdx.x);
      const int row = v >> 2, t = row / kNB, o = row % kNB;
      const int nt = (o >> 2) & 1, m = 4 * (o >> 3) + (o & 3);   // frag_out(m, nt) == o
      if (v < kWVec) ws[buf][(2 * t + nt) * 64 + 16 * (v & 3) + m] = wreg[k];
    }
  };

  // ---- input rows ----
  struct Unit {            // a tile's step of 32 channels
    const char *base;      // the image's first row in the step's source
    int rowbytes, up, y0;
    bool valid;
    uint32_t oc, oe;       // the lane's offsets in a row: its pixel, the edge pixel
  };
  auto make_unit = [&](int grp, int c0) {
    Unit u;
    const TileAt t = tile_at<R>(grp * kWaves + wave, ntiles, tiles_x, tiles_y);
    const bool first_src = c0 < src.ca;
    const int C = first_src ? src.ca : src.cb, c = first_src ? c0 : c0 - src.ca;
    u.up = first_src ? src.up : 0;
    u.rowbytes = (W >> u.up) * C * 2;
    u.base = reinterpret_cast<const char *>(first_src ? src.a : src.b) +
             t.b * (H >> u.up) * static_cast<long>(u.rowbytes);
    u.y0 = t.y0;
    u.valid = t.valid && grp < g1;
    const bool cok = c + 8 * g < C;
    const int xc = (t.x0 + r) >> u.up, xe = (r == 0 ? t.x0 - 1 : t.x0 + 16) >> u.up;
    u.oc = cok ? static_cast<uint32_t>(xc * C + c + 8 * g) * 2u : kOob;
    u.oe = cok && (r == 0 || r == 15) ? static_cast<uint32_t>(xe * C + c + 8 * g) * 2u : kOob;
    return u;
  };
  // rows in flight: row p sits in slot p % kRing
  constexpr int kRing = R == 8 ? 5 : R + 2;
  static_assert((R + 2) % kRing == 0, "slots line up from step to step");
  u32x4 pc[kRing], pe[kRing];
  auto load_row = [&](const Unit &u, int p) {
    const int yy = u.y0 - 1 + p;
    const bool ok = u.valid && static_cast<unsigned>(yy) < static_cast<unsigned>(H);
    const char *row = u.base + static_cast<long>(ok ? yy >> u.up : 0) * u.rowbytes;
    pc[p % kRing] = load_px(row, ok ? u.rowbytes : 0, u.oc);
    pe[p % kRing] = load_px(row, ok ? u.rowbytes : 0, u.oe);
  };

  f32x4 acc[R][2];
#pragma unroll
  for (int y = 0; y < R; y++) acc[y][0] = acc[y][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch_weights(0);
  Unit cur = make_unit(first, 0);
#pragma unroll
  for (int p = 0; p < kRing; p++) load_row(cur, p);
  stage_weights(0);
  __syncthreads();
  u32x4 w[9][2];
#pragma unroll
  for (int f = 0; f < kWFrags; f++) w[f >> 1][f & 1] = ws[0][f * 64 + lane];
  int buf = 0;
  for (int grp = first; grp < g1; grp += per) {
    for (int cs = 0; cs < csteps; cs++) {
      const bool last = cs + 1 == csteps;
      const bool more = !last || grp + per < g1;
      const int cnext = last ? 0 : (cs + 1) * kKC;
      const Unit next = make_unit(last ? grp + per : grp, cnext);
      if (csteps > 1 && more) fetch_weights(cnext);
#pragma unroll
      for (int p = 0; p < R + 2; p++) {
        const u32x4 c = pc[p % kRing], e = pe[p % kRing];
        const u32x4 f[3] = {from_left(c, e), c, from_right(c, e)};
        if (p + kRing < R + 2) load_row(cur, p + kRing);
        else load_row(next, p + kRing - (R + 2));
#pragma unroll
        for (int dx = 0; dx < 3; dx++)
#pragma unroll
          for (int dy = 0; dy < 3; dy++) {
            const int y = p - dy;
            if (y < 0 || y >= R) continue;
#pragma unroll
            for (int nt = 0; nt < 2; nt++)
              acc[y][nt] = mfma16(w[3 * dy + dx][nt], f[dx], acc[y][nt]);
          }
      }
      cur = next;
      if (csteps > 1 && more) {
        // the other buffer's readers passed the previous barrier; only LDS is
        // waited for, the rows requested above stay in flight
        buf ^= 1;
        stage_weights(buf);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int f = 0; f < kWFrags; f++) w[f >> 1][f & 1] = ws[buf][f * 64 + lane];
      }
    }
    store_tile<R>(acc, tile_at<R>(grp * kWaves + wave, ntiles, tiles_x, tiles_y), dst, bias, relu,
                  n0, nout, H, W);
#pragma unroll
    for (int y = 0; y < R; y++) acc[y][0] = acc[y][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// Few tiles: one wave per workgroup, 16 columns x 2 rows x 32 outputs, no LDS,
// the loop over (channel step, tap) or, for levels smaller than 8 x 16, over (tap,
// channel step), with kAhead iterations' operands in flight.
template <bool kTapOuter>
__global__ __launch_bounds__(64) void k_conv_small(ConvSrc src, const uint16_t *__restrict__ wt,
                                                   const float *__restrict__ bias, int relu,
                                                   ConvDst dst, int nout, int H, int W,
                                                   int tiles_x, int tiles_y, int ntiles) {
  constexpr int R = 2, kAhead = 9;
  const int lane = threadIdx.x, g = lane >> 4, r = lane & 15;
  const int n0 = blockIdx.y * kNB;
  const TileAt t = tile_at<R>(blockIdx.x, ntiles, tiles_x, tiles_y);
  const int cin = src.ca + src.cb, csteps = (cin + kKC - 1) / kKC, steps = 9 * csteps;
  // The wave is alone on its SIMD and bound by its instructions (12, 15 or 18
  // iterations in flight are no faster than 9), so what a lane
  // adds to an address is computed here, once, and the rest is the loads'
  // scalar offset (8 x 8 levels of 160 channels: 12.6 us with every
  // load's address computed anew, 9.5 now).  Columns beyond the image and
  // channels beyond cin (the network's input has 8) lie out of range.
  struct Side {
    const char *rows;      // the rows the tile reads (fs_conv_rows.h)
    int bytes, up;
    uint32_t rowbytes, skip;
    uint32_t x[3];
  };
  auto side_of = [&](const uint16_t *base, int C, int up) {
    Side q;
    const int rowbytes = (W >> up) * C * 2;
    const fs::ConvRows at = fs::conv_rows(t.y0, R, H, up, rowbytes);
    q.up = up;
    q.rowbytes = static_cast<uint32_t>(rowbytes);
    q.skip = at.skip;
    q.bytes = static_cast<int>(at.bytes);
    q.rows = reinterpret_cast<const char *>(base) + t.b * (H >> up) * static_cast<long>(rowbytes) +
             at.start;
#pragma unroll
    for (int dx = 0; dx < 3; dx++) {
      const int x = t.x0 + r + dx - 1;
      q.x[dx] = static_cast<unsigned>(x) < static_cast<unsigned>(W) && 8 * g < C
                    ? static_cast<uint32_t>((x >> up) * C + 8 * g) * 2u
                    : kOob;
    }
    return q;
  };
  const Side sa = side_of(src.a, src.ca, src.up), sb = side_of(src.b, src.cb, 0);
  uint32_t wo[2];
#pragma unroll
  for (int nt = 0; nt < 2; nt++)
    wo[nt] = 8 * g < cin ? static_cast<uint32_t>((n0 + frag_out(r, nt)) * cin + 8 * g) * 2u : kOob;
  u32x4 px[kAhead][R], wv[kAhead][2];
  int lt = 0, lc = 0;    // tap and first channel of the next iteration to load
  auto load = [&](int slot) {
    // iteration s is in slot s % 9; past the last one the first ones come again
    const int tt = kTapOuter ? lt : slot;
    const bool first_src = lc < src.ca;
    const char *rows = first_src ? sa.rows : sb.rows;
    const int bytes = first_src ? sa.bytes : sb.bytes, up = first_src ? sa.up : 0;
    const uint32_t rowbytes = first_src ? sa.rowbytes : sb.rowbytes;
    const uint32_t skip = first_src ? sa.skip : sb.skip;
    const int c2 = 2 * (first_src ? lc : lc - src.ca);
    const int dy = tt / 3, dx = tt - 3 * dy;
    // selects by hand: an index into sa.x would put it into memory
    const uint32_t x0 = first_src ? sa.x[0] : sb.x[0], x1 = first_src ? sa.x[1] : sb.x[1];
    const uint32_t x2 = first_src ? sa.x[2] : sb.x[2];
    const uint32_t x = dx == 0 ? x0 : dx == 1 ? x1 : x2;
#pragma unroll
    for (int y = 0; y < R; y++) {
      const int yy = t.y0 + y + dy - 1;
      const bool in = static_cast<unsigned>(yy) < static_cast<unsigned>(H);
      px[slot][y] = load_px_at(
          rows, in ? bytes : 0, x,
          in ? static_cast<int>(fs::conv_row_offset(yy, up, rowbytes, skip)) + c2 : 0);
    }
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
      wv[slot][nt] = load_px_at(reinterpret_cast<const char *>(wt), 9 * nout * cin * 2, wo[nt],
                                (tt * nout * cin + lc) * 2);
    if (kTapOuter) {
      lc += kKC;
      if (lc >= cin) {
        lc = 0;
        lt = lt == 8 ? 0 : lt + 1;
      }
    } else if (slot == 8) {
      lc = lc + kKC >= cin ? 0 : lc + kKC;
    }
  };
  f32x4 acc[R][2];
#pragma unroll
  for (int y = 0; y < R; y++) acc[y][0] = acc[y][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < kAhead; d++) load(d);
  for (int s = 0; s < steps; s += kAhead) {   // steps is a multiple of kAhead
#pragma unroll
    for (int d = 0; d < kAhead; d++) {
#pragma unroll
      for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int y = 0; y < R; y++) acc[y][nt] = mfma16(wv[d][nt], px[d][y], acc[y][nt]);
      load(d);
    }
  }
  store_tile<R>(acc, t, dst, bias, relu, n0, nout, H, W);
}

// ---------------------------------------------------------------------------
// Weight gradient of a 3x3 convolution, split over pixel chunks:
//   part[chunk][t][co][ci] = sum_{p in chunk} dz[p][co] * x[p + off_t][ci]
// GEMM with M = co, N = ci (64 x 64 per workgroup, 32 x 32 per wave),
// K = pixels in steps of 32, both operands staged through LDS transposed so
// that each lane reads 8 consecutive pixels of one channel.
// ---------------------------------------------------------------------------
constexpr int kDwStride = 40;   // LDS row: 32 pixels + 8 pad (80 bytes)

__global__ __launch_bounds__(256) void k_conv3x3_dw(const uint16_t *__restrict__ dz, int cout,
                                                    ConvSrc src, float *__restrict__ part, int H,
                                                    int W, long chunk_pix, long M) {
  __shared__ __attribute__((aligned(16))) uint16_t As[64 * kDwStride];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[64 * kDwStride];
  const int cin = src.ca + src.cb;
  const int tiles_ci = (cin + 63) / 64;
  const int co0 = (blockIdx.x / tiles_ci) * 64, ci0 = (blockIdx.x % tiles_ci) * 64;
  const int t = blockIdx.y, chunk = blockIdx.z;
  const int dy = t / 3 - 1, dx = t % 3 - 1;
  const long k0 = chunk * chunk_pix, k1 = min(M, k0 + chunk_pix);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int rb = (wave >> 1) * 32, cb = (wave & 1) * 32;
  // loader: pixel lp = tid/8, channels 8*(tid%8) .. +7
  const int lp = threadIdx.x >> 3, lc = (threadIdx.x & 7) * 8;
  const bool first_src = ci0 + lc < src.ca;
  const int up = first_src ? src.up : 0, xC = first_src ? src.ca : src.cb;
  const uint16_t *const x = first_src ? src.a + ci0 + lc : src.b + (ci0 + lc - src.ca);
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int c = 0; c < 2; c++) acc[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (long kp = k0; kp < k1; kp += 32) {
    const long p = kp + lp;
    uint4 zv = make_uint4(0u, 0u, 0u, 0u), xv = make_uint4(0u, 0u, 0u, 0u);
    if (p < k1) {
      if (co0 + lc < cout) zv = *reinterpret_cast<const uint4 *>(dz + p * cout + co0 + lc);
      const int px = static_cast<int>(p % W);
      const long pq = p / W;
      const int py = static_cast<int>(pq % H);
      const long pb = pq / H;
      const int yy = py + dy, xx = px + dx;
      if (ci0 + lc < cin && yy >= 0 && yy < H && xx >= 0 && xx < W)
        xv = *reinterpret_cast<const uint4 *>(
            x + ((pb * (H >> up) + (yy >> up)) * (W >> up) + (xx >> up)) * xC);
    }
    const uint16_t *zs = reinterpret_cast<const uint16_t *>(&zv);
    const uint16_t *xs = reinterpret_cast<const uint16_t *>(&xv);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      As[(lc + j) * kDwStride + lp] = zs[j];
      Bs[(lc + j) * kDwStride + lp] = xs[j];
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 2; a++) {
      const uint4 av = *reinterpret_cast<const uint4 *>(&As[(rb + a * 16 + r) * kDwStride + 8 * g]);
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const uint4 bv = *reinterpret_cast<const uint4 *>(&Bs[(cb + c * 16 + r) * kDwStride + 8 * g]);
        acc[a][c] = mfma16(av, bv, acc[a][c]);
      }
    }
    __syncthreads();
  }
  float *dst = part + (static_cast<long>(chunk) * 9 + t) * cout * cin;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int co = co0 + rb + a * 16 + 4 * g + i, ci = ci0 + cb + c * 16 + r;
        if (co < cout && ci < cin) dst[static_cast<long>(co) * cin + ci] = acc[a][c][i];
      }
}

// dw[i] = sum over chunks of part[chunk][i]
__global__ __launch_bounds__(256) void k_reduce_chunks(const float *__restrict__ part,
                                                       float *__restrict__ dw, long n,
                                                       int nchunks) {
  for (long i = blockIdx.x * 256l + threadIdx.x; i < n; i += gridDim.x * 256l) {
    float s = 0.f;
    for (int c = 0; c < nchunks; c++) s += part[c * n + i];
    dw[i] = s;
  }
}

// ---------------------------------------------------------------------------
// Weight gradient with all nine taps per wave:
//   part[chunk][t][co][ci] = sum over the chunk's pixels of
//                            dz[p][co] * x[p + off_t][ci]
// K = pixels: a step is one row of two strips (16 columns x R rows of an
// image), 32 pixels.  Both tensors go to LDS as they lie in memory, [pixel]
// [channel]; ds_read_b64_tr_b16 hands each lane four consecutive pixels of its
// channel, so nothing is transposed in registers and every tap reads the same
// patch at its own pixel offset.  A wave owns 32 outputs x 16 inputs x 9 taps
// and walks down the rows: the gradient rows of the last three are kept, so a
// patch row's three column shifts are read once for nine taps (10 reads for 18
// MFMAs).  A workgroup's four waves take NC blocks of 32 outputs x two halves
// of 32 inputs, NK pairs of strips at a time.  LDS rows are padded so that the
// 32-byte pieces of a read fall on different banks.
// With db, the workgroups of the first input block also add the bias gradient
// sum_p dz[p][co] of their pixels to db.  Needs H % R == 0, W % 16 == 0, cout %
// (32 * NC) == 0, cin % 8 == 0, and ca % 32 == 0 where there are two sources.
//
// With 8 x 8 transposes in registers, three shifted copies of the patch and
// three waves per workgroup, the weight gradients took 1.95 ms of the backward
// pass of 32 samples of 256 x 256 (321 TFLOP/s); they take 1.20 (523).  <2, 1> moves
// its bytes at 5.5 TB/s, a copy's rate (every block of inputs reads the gradients
// again); <1, 2> is bound by no one unit (matrix units busy 18% of the cycles, LDS
// 24%, 3.8 TB/s).
// ---------------------------------------------------------------------------
typedef short i16x4 __attribute__((ext_vector_type(4)));
constexpr int kDwThreads = 256;
template <int NC, int NK>
struct DwShape {
  static constexpr int R = NK == 1 ? 8 : 4;          // rows of a strip
  static constexpr int kXPix = (R + 2) * 18, kZPix = R * 16;
  static constexpr int kXS = 32 + 16, kZS = 32 * NC + 16;   // halfwords per pixel in LDS
  static constexpr int kStrips = 2 * NK;
};

// 8 pixels p .. p+7 of one channel per lane, from two transposing reads: `at` is
// the lane's place in the first (pixel (lane % 16) / 4, channels 4 * (lane % 4)
// ..), the second lies 4 pixels on.
__device__ __forceinline__ u32x4 read_pixels(const uint16_t *at, int stride) {
  typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
  uint16_t *const p = const_cast<uint16_t *>(at);
  const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p));
  const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p + 4 * stride));
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  const u32x2 l = __builtin_bit_cast(u32x2, lo), h = __builtin_bit_cast(u32x2, hi);
  return u32x4{l.x, l.y, h.x, h.y};
}

template <int NC, int NK>
__global__ __launch_bounds__(kDwThreads, 2) void k_conv_dw(
    const uint16_t *__restrict__ dz, int cout, ConvSrc src, float *__restrict__ part,
    float *__restrict__ db, int H, int W, long strips, long units, int units_per_chunk,
    int ci_blocks) {
  using S = DwShape<NC, NK>;
  constexpr int R = S::R;
  static_assert(2 * NC * NK == 4, "four waves");
  __shared__ __attribute__((aligned(16))) uint16_t xs[S::kStrips * S::kXPix * S::kXS];
  __shared__ __attribute__((aligned(16))) uint16_t zs[S::kStrips * S::kZPix * S::kZS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int cih = wave & 1, coh = NC == 2 ? wave >> 1 : 0, kh = NK == 2 ? wave >> 1 : 0;
  const int co0 = (blockIdx.x / ci_blocks) * 32 * NC, ci0 = (blockIdx.x % ci_blocks) * 32;
  const int cin = src.ca + src.cb;
  // the block's 32 inputs lie in one of the two sources
  const bool first_src = ci0 < src.ca;
  const int up = first_src ? src.up : 0, xC = first_src ? src.ca : src.cb;
  const uint16_t *const x = first_src ? src.a + ci0 : src.b + (ci0 - src.ca);
  const int xch = min(32, cin - ci0);
  const int strips_x = W / 16, strips_img = (H / R) * strips_x;
  const long u0 = static_cast<long>(blockIdx.y) * units_per_chunk;
  const long u1 = min(units, u0 + units_per_chunk);

  // staging registers: 16-byte vectors of 8 channels
  constexpr int kXVec = S::kStrips * S::kXPix * 4, kZVec = S::kStrips * S::kZPix * 4 * NC;
  constexpr int kXPer = (kXVec + kDwThreads - 1) / kDwThreads, kZPer = kZVec / kDwThreads;
  static_assert(kZVec % kDwThreads == 0, "whole vectors per thread");
  u32x4 xv[kXPer], zv[kZPer];
  auto fetch = [&](long unit) {
    long base[S::kStrips];       // image, and the strip's first pixel in it
    int sy[S::kStrips], sx[S::kStrips];
    bool ok[S::kStrips];
#pragma unroll
    for (int j = 0; j < S::kStrips; j++) {
      const long s = unit * S::kStrips + j;
      ok[j] = s < strips;
      const long q = ok[j] ? s : 0;
      base[j] = q / strips_img;
      const int t = static_cast<int>(q - base[j] * strips_img);
      sy[j] = (t / strips_x) * R;
      sx[j] = (t % strips_x) * 16;
    }
#pragma unroll
    for (int k = 0; k < kXPer; k++) {
      const int v = k * kDwThreads + static_cast<int>(threadIdx.x);
      const int j = v / (4 * S::kXPix), e = v - j * 4 * S::kXPix;
      const int pix = e >> 2, c = 8 * (e & 3);
      const int py = pix / 18, px = pix - 18 * py;
      int yy = 0, xx = 0;
      long b = 0;
      bool in = false;
#pragma unroll
      for (int q = 0; q < S::kStrips; q++)
        if (j == q) {
          yy = sy[q] - 1 + py;
          xx = sx[q] - 1 + px;
          b = base[q];
          in = ok[q];
        }
      in = in && v < kXVec && c < xch && static_cast<unsigned>(yy) < static_cast<unsigned>(H) &&
           static_cast<unsigned>(xx) < static_cast<unsigned>(W);
      xv[k] = u32x4{0u, 0u, 0u, 0u};
      if (in)
        xv[k] = *reinterpret_cast<const u32x4 *>(
            x + ((b * (H >> up) + (yy >> up)) * (W >> up) + (xx >> up)) * xC + c);
    }
#pragma unroll
    for (int k = 0; k < kZPer; k++) {
      const int v = k * kDwThreads + static_cast<int>(threadIdx.x);
      const int j = v / (4 * NC * S::kZPix), e = v - j * 4 * NC * S::kZPix;
      const int pix = e / (4 * NC), c = 8 * (e % (4 * NC));
      int yy = 0, xx = 0;
      long b = 0;
      bool in = false;
#pragma unroll
      for (int q = 0; q < S::kStrips; q++)
        if (j == q) {
          yy = sy[q] + pix / 16;
          xx = sx[q] + pix % 16;
          b = base[q];
          in = ok[q];
        }
      zv[k] = u32x4{0u, 0u, 0u, 0u};
      if (in)
        zv[k] = *reinterpret_cast<const u32x4 *>(dz + ((b * H + yy) * W + xx) * cout + co0 + c);
    }
  };
  const bool bias = db != nullptr && blockIdx.x % ci_blocks == 0;
  float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // of this thread's 8 outputs
  auto stage = [&]() {
#pragma unroll
    for (int k = 0; k < kXPer; k++) {
      const int v = k * kDwThreads + static_cast<int>(threadIdx.x);
      if (v < kXVec) *reinterpret_cast<u32x4 *>(&xs[(v >> 2) * S::kXS + 8 * (v & 3)]) = xv[k];
    }
#pragma unroll
    for (int k = 0; k < kZPer; k++) {
      const int v = k * kDwThreads + static_cast<int>(threadIdx.x);
      *reinterpret_cast<u32x4 *>(&zs[(v / (4 * NC)) * S::kZS + 8 * (v % (4 * NC))]) = zv[k];
      if (bias) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          bsum[2 * e] += bf_lo(zv[k][e]);
          bsum[2 * e + 1] += bf_hi(zv[k][e]);
        }
      }
    }
  };

  f32x4 acc[9][2];
#pragma unroll
  for (int t = 0; t < 9; t++) acc[t][0] = acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the lane's place in a transposing read: strip g / 2, pixel 8 * (g % 2) + r / 4
  const int strip = 2 * kh + (g >> 1), pix = 8 * (g & 1) + (r >> 2);
  const uint16_t *const xl = &xs[(strip * S::kXPix + pix) * S::kXS + 16 * cih + 4 * (r & 3)];
  const uint16_t *const zl = &zs[(strip * S::kZPix + pix) * S::kZS + 32 * coh + 4 * (r & 3)];
  // this lane's sums in part, by 32-bit offsets from the chunk's (inputs beyond cin:
  // beyond them all)
  const __amdgpu_buffer_rsrc_t sums = __builtin_amdgcn_make_buffer_rsrc(
      part + static_cast<long>(blockIdx.y) * 9 * cout * cin, 0, 36 * cout * cin, kRsrc);
  const uint32_t sum_at = ci0 + 16 * cih + r < cin
                              ? static_cast<uint32_t>((co0 + 32 * coh + 4 * g) * cin + ci0 +
                                                      16 * cih + r) * 4u
                              : kOob;
  auto each_sum = [&](auto f) {
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int i = 0; i < 4; i++) f(t, h, i, 4 * (t * cout + 16 * h + i) * cin);
  };
  auto store_sum = [&](int t, int h, int i, int at) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[t][h][i]), sums,
                                          static_cast<int>(sum_at), at, 0);
  };
  // Where one wave sums all of the workgroup's pixels, its sums go to memory
  // halfway and start again from zero: an accumulator's rounding error grows with
  // its sum's length (against sums in 32 times as many chunks, the 288 -> 128 layer
  // of 32 samples of 256 x 256 is off by 2.4e-7 of its norm in one go, by 2.0e-7
  // this way).  It costs the loss and gradients of that batch 2.5%.
  const long half = NK == 1 && u1 - u0 > 1 ? u0 + (u1 - u0 + 1) / 2 : u1;
  if (u0 < u1) fetch(u0);
  for (long unit = u0; unit < u1; unit++) {
    if (NK == 1 && unit == half) {
      each_sum(store_sum);
#pragma unroll
      for (int t = 0; t < 9; t++) acc[t][0] = acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    stage();
    __syncthreads();
    if (unit + 1 < u1) fetch(unit + 1);
    u32x4 a[3][2];
#pragma unroll
    for (int pr = 0; pr < R + 2; pr++) {
      if (pr < R) {
#pragma unroll
        for (int h = 0; h < 2; h++)
          a[pr % 3][h] = read_pixels(zl + pr * 16 * S::kZS + 16 * h, S::kZS);
      }
#pragma unroll
      for (int dx = 0; dx < 3; dx++) {
        const u32x4 bv = read_pixels(xl + (pr * 18 + dx) * S::kXS, S::kXS);
#pragma unroll
        for (int dy = 0; dy < 3; dy++) {
          const int y = pr - dy;
          if (y < 0 || y >= R) continue;
#pragma unroll
          for (int h = 0; h < 2; h++)
            acc[3 * dy + dx][h] = mfma16(a[y % 3][h], bv, acc[3 * dy + dx][h]);
        }
      }
    }
    __syncthreads();
  }
  // the two halves of the pixels, added up in LDS (free after the last barrier)
  if constexpr (NK == 2) {
    f32x4 *const half = reinterpret_cast<f32x4 *>(xs);
    static_assert(sizeof(xs) >= 2 * 18 * 64 * sizeof(f32x4), "room for one half's sums");
    if (kh == 1) {
#pragma unroll
      for (int t = 0; t < 9; t++)
#pragma unroll
        for (int h = 0; h < 2; h++) half[((cih * 9 + t) * 2 + h) * 64 + lane] = acc[t][h];
    }
    __syncthreads();
    if (kh == 0) {
#pragma unroll
      for (int t = 0; t < 9; t++)
#pragma unroll
        for (int h = 0; h < 2; h++) acc[t][h] += half[((cih * 9 + t) * 2 + h) * 64 + lane];
    }
  }
  if (bias) {
    // threads with the same 8 outputs lie 4 * NC apart
    float *const red = reinterpret_cast<float *>(zs);
#pragma unroll
    for (int e = 0; e < 8; e++) red[threadIdx.x * 8 + e] = bsum[e];
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < 32 * NC) {
      const int c8 = threadIdx.x / 8, e = threadIdx.x % 8;
      float sum = 0.f;
      for (int q = c8; q < kDwThreads; q += 4 * NC) sum += red[q * 8 + e];
      atomicAdd(&db[co0 + threadIdx.x], sum);
    }
  }
  if (half < u1)
    each_sum([&](int t, int h, int i, int at) {
      acc[t][h][i] += __uint_as_float(
          __builtin_amdgcn_raw_buffer_load_b32(sums, static_cast<int>(sum_at), at, 0));
    });
  if (kh == 0) each_sum(store_sum);
}

// dw[i] = sum over chunks of part[chunk][i]; 64 elements x 16 chunk lanes per
// workgroup, the chunk lanes combined in LDS.  Bound by the latency of a lane's
// loads: four in flight measured 7.8 us a layer against 10.5 one after another.
__global__ __launch_bounds__(1024) void k_reduce_chunks_wide(const float *__restrict__ part,
                                                             float *__restrict__ dw, long n,
                                                             int nchunks) {
  __shared__ float red[16][64];
  const int e = threadIdx.x & 63, cl = threadIdx.x >> 6;
  const long i = static_cast<long>(blockIdx.x) * 64 + e;
  float s = 0.f;
  if (i < n) {
    const float *p = part + i;
    int c = cl;
    for (; c + 48 < nchunks; c += 64) {   // four loads in flight
      const float a = p[static_cast<long>(c) * n], b = p[static_cast<long>(c + 16) * n];
      const float d = p[static_cast<long>(c + 32) * n], f = p[static_cast<long>(c + 48) * n];
      s += (a + b) + (d + f);
    }
    for (; c < nchunks; c += 16) s += p[static_cast<long>(c) * n];
  }
  red[cl][e] = s;
  __syncthreads();
  if (cl == 0 && i < n) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 16; k++) t += red[k][e];
    dw[i] = t;
  }
}

// db[c] += sum_p dz[p][c] over the block's pixel range; thread t sums the
// 8-channel group t % C8 over every (256 / C8)-th pixel, C % 8 == 0, C <= 512
__global__ __launch_bounds__(256) void k_bias_grad(const uint16_t *__restrict__ dz, int C,
                                                   float *__restrict__ db, long M,
                                                   long chunk_pix) {
  __shared__ float red[512];
  for (int c = threadIdx.x; c < C; c += 256) red[c] = 0.f;
  __syncthreads();
  const int C8 = C / 8, lanes = 256 / C8;
  const long p0 = blockIdx.x * chunk_pix, p1 = min(M, p0 + chunk_pix);
  if (static_cast<int>(threadIdx.x) < lanes * C8) {
    const int c8 = threadIdx.x % C8, pl = threadIdx.x / C8;
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (long p = p0 + pl; p < p1; p += lanes) {
      const uint4 v = *reinterpret_cast<const uint4 *>(dz + p * C + 8 * c8);
      const uint16_t *h = reinterpret_cast<const uint16_t *>(&v);
#pragma unroll
      for (int k = 0; k < 8; k++) s[k] += bf2f(h[k]);
    }
#pragma unroll
    for (int k = 0; k < 8; k++) atomicAdd(&red[8 * c8 + k], s[k]);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < C; c += 256) atomicAdd(&db[c], red[c]);
}

// gradient of the pooling, added to the skip connection's:
// dx[b,y,x,c] = dx[b,y,x,c] + dy[b,y/2,x/2,c] / 4 where act[b,y,x,c] > 0, else 0
// (act: the pooled tensor, a ReLU's output)
__global__ __launch_bounds__(256) void k_pool_grad(const uint16_t *__restrict__ dy,
                                                   uint16_t *__restrict__ dx,
                                                   const uint16_t *__restrict__ act, int B, int H,
                                                   int W, int C) {
  const int C8 = C / 8;
  const long n = static_cast<long>(B) * H * W * C8;
  for (long i = blockIdx.x * 256l + threadIdx.x; i < n; i += gridDim.x * 256l) {
    const int c8 = static_cast<int>(i % C8);
    const long q = i / C8;
    const int x = static_cast<int>(q % W);
    const long q2 = q / W;
    const int y = static_cast<int>(q2 % H);
    const long b = q2 / H;
    const long src = ((b * (H / 2) + y / 2) * (W / 2) + x / 2) * C + 8 * c8;
    const u32x4 v = *reinterpret_cast<const u32x4 *>(dy + src);
    u32x4 *const dst = reinterpret_cast<u32x4 *>(dx + q * C + 8 * c8);
    const u32x4 e = *dst, m = *reinterpret_cast<const u32x4 *>(act + q * C + 8 * c8);
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; k++)
      o[k] = relu_mask(pack_bf(bf_lo(e[k]) + 0.25f * bf_lo(v[k]), bf_hi(e[k]) + 0.25f * bf_hi(v[k])),
                       m[k]);
    *dst = o;
  }
}

// network input: [terrain, p0, p1, p2, 0, 0, 0, 0] per pixel
// (terrain_stride 0: one terrain shared by the batch)
__global__ __launch_bounds__(256) void k_pack_input(const float *__restrict__ terrain,
                                                    const float *__restrict__ params,
                                                    uint16_t *__restrict__ x, int B, long HW,
                                                    long terrain_stride) {
  for (long i = blockIdx.x * 256l + threadIdx.x; i < B * HW; i += gridDim.x * 256l) {
    const long b = i / HW;
    uint16_t o[8] = {f2bf(terrain[b * terrain_stride + i % HW]), f2bf(params[3 * b]),
                     f2bf(params[3 * b + 1]),
                     f2bf(params[3 * b + 2]), 0, 0, 0, 0};
    *reinterpret_cast<uint4 *>(x + i * 8) = *reinterpret_cast<const uint4 *>(o);
  }
}

// sq[b] += sum over the interior (rings 0, 1 excluded) of (yhat - t)^2 for
// the batch's samples, against one target t of H x W
__global__ __launch_bounds__(256) void k_sq_misfit(const float *__restrict__ yhat,
                                                   const float *__restrict__ t,
                                                   float *__restrict__ sq, int H, int W) {
  __shared__ float red;
  if (threadIdx.x == 0) red = 0.f;
  __syncthreads();
  const long HW = static_cast<long>(H) * W;
  const int b = blockIdx.y;
  float s = 0.f;
  for (long i = blockIdx.x * 256l + threadIdx.x; i < HW; i += gridDim.x * 256l) {
    const int x = static_cast<int>(i % W), y = static_cast<int>(i / W);
    if (x < 2 || y < 2 || x >= W - 2 || y >= H - 2) continue;
    const float d = yhat[b * HW + i] - t[i];
    s += d * d;
  }
  atomicAdd(&red, s);
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(&sq[b], red);
}

// head: yhat[p] = hb + sum_c hw[c] * f[p][c], C = 32
__global__ __launch_bounds__(256) void k_head(const uint16_t *__restrict__ f,
                                              const float *__restrict__ hw,
                                              const float *__restrict__ hb,
                                              float *__restrict__ yhat, long M) {
  for (long p = blockIdx.x * 256l + threadIdx.x; p < M; p += gridDim.x * 256l) {
    float s = hb[0];
#pragma unroll
    for (int c8 = 0; c8 < 4; c8++) {
      const uint4 v = *reinterpret_cast<const uint4 *>(f + p * 32 + 8 * c8);
      const uint16_t *h = reinterpret_cast<const uint16_t *>(&v);
#pragma unroll
      for (int k = 0; k < 8; k++) s += hw[8 * c8 + k] * bf2f(h[k]);
    }
    yhat[p] = s;
  }
}

// loss = mean (yhat - t)^2 over M pixels; gy = 2 (yhat - t) / M; head
// gradients; df[p][c] = gy[p] * hw[c] where f[p][c] > 0, else 0 (f is a ReLU's
// output).  *loss += loss, gh[0..31] += dhw, gh[32] += dhb.
// Four lanes per pixel, 8 channels each: a wave reads and writes whole runs of
// memory, and the sums meet by shuffles, then once per workgroup in LDS.  (One
// lane per pixel and 34 LDS atomics per thread on the same 34 words: 194 us for
// 32 samples of 256 x 256 against 71; the 285 MB it moves take 57 at 5 TB/s.)
__global__ __launch_bounds__(256) void k_head_grad(const uint16_t *__restrict__ f,
                                                   const float *__restrict__ hw,
                                                   const float *__restrict__ yhat,
                                                   const float *__restrict__ tgt,
                                                   uint16_t *__restrict__ df,
                                                   float *__restrict__ loss,
                                                   float *__restrict__ gh, long M) {
  __shared__ float red[4][34];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c0 = 8 * (lane & 3);
  float w[8], gw[8], l = 0.f, gb = 0.f;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    w[k] = hw[c0 + k];
    gw[k] = 0.f;
  }
  const float inv = 1.0f / static_cast<float>(M);
  for (long q = blockIdx.x * 256l + threadIdx.x; q < 4 * M; q += gridDim.x * 256l) {
    const long p = q >> 2;
    const float e = yhat[p] - tgt[p];
    const u32x4 v = *reinterpret_cast<const u32x4 *>(f + p * 32 + c0);
    const float gy = 2.0f * e * inv;
    if (c0 == 0) {
      l += e * e * inv;
      gb += gy;
    }
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      gw[2 * k] += gy * bf_lo(v[k]);
      gw[2 * k + 1] += gy * bf_hi(v[k]);
      o[k] = relu_mask(pack_bf(gy * w[2 * k], gy * w[2 * k + 1]), v[k]);
    }
    *reinterpret_cast<u32x4 *>(df + p * 32 + c0) = o;
  }
#pragma unroll
  for (int d = 4; d < 64; d <<= 1) {
    l += __shfl_xor(l, d);
    gb += __shfl_xor(gb, d);
#pragma unroll
    for (int k = 0; k < 8; k++) gw[k] += __shfl_xor(gw[k], d);
  }
  if (lane < 4) {
#pragma unroll
    for (int k = 0; k < 8; k++) red[wave][c0 + k] = gw[k];
    if (lane == 0) {
      red[wave][32] = gb;
      red[wave][33] = l;
    }
  }
  __syncthreads();
  if (threadIdx.x < 34) {
    const float s = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] +
                    red[3][threadIdx.x];
    atomicAdd(threadIdx.x < 33 ? &gh[threadIdx.x] : loss, s);
  }
}

// Adam (Kingma & Ba 2015) on the FP32 masters
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ w, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v,
                                              long n, float lr, float b1, float b2, float eps,
                                              float c1, float c2) {
  for (long i = blockIdx.x * 256l + threadIdx.x; i < n; i += gridDim.x * 256l) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// BF16 copies of one conv layer's weights W[t][co][ci]:
//   wf[t][co][ci] = W[t][co][ci];   wb[t][ci][co] = W[8-t][co][ci]
__global__ __launch_bounds__(256) void k_pack_weights(const float *__restrict__ w,
                                                      uint16_t *__restrict__ wf,
                                                      uint16_t *__restrict__ wb, int cout,
                                                      int cin) {
  const long n = 9l * cout * cin;
  for (long i = blockIdx.x * 256l + threadIdx.x; i < n; i += gridDim.x * 256l) {
    const int ci = static_cast<int>(i % cin);
    const long q = i / cin;
    const int co = static_cast<int>(q % cout);
    const int t = static_cast<int>(q / cout);
    const uint16_t v = f2bf(w[i]);
    wf[i] = v;
    wb[(static_cast<long>(8 - t) * cin + ci) * cout + co] = v;
  }
}

__global__ __launch_bounds__(256) void k_fill_f32(float *p, long n, float v) {
  for (long i = blockIdx.x * 256l + threadIdx.x; i < n; i += gridDim.x * 256l) p[i] = v;
}

}  // namespace

// ===========================================================================
// host side
// ===========================================================================
namespace {

struct Conv {
  int cin, cout, level;        // level: resolution H>>level
  size_t woff, boff;           // offsets into the parameter vector
  uint16_t *wf = nullptr, *wb = nullptr;
};

struct Tensor {
  uint16_t *d = nullptr;   // device, max_batch x (H>>level) x (W>>level) x C
  int C = 0, level = 0;
};

}  // namespace

struct fs_unet {
  int H = 0, W = 0, max_batch = 0, device = 0;
  hipStream_t stream = nullptr;
  hipStream_t copy = nullptr;             // host copies beside the kernels
  hipEvent_t copy_ev[2] = {nullptr, nullptr};
  std::vector<Conv> conv;   // 14 layers
  size_t nparam = 0, head_w = 0, head_b = 0;
  float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;   // FP32 params, grads, Adam
  float *part = nullptr;
  size_t part_n = 0;
  // activations and their gradients
  Tensor x0, e_a[kLevels], e[kLevels], p[kLevels - 1], d_a[kLevels - 1], d[kLevels - 1];
  // gradients of the convolutions' outputs before their ReLU; gp: of the
  // pooled tensors
  Tensor ge_a[kLevels], ge[kLevels], gp[kLevels - 1], gd_a[kLevels - 1], gd[kLevels - 1];
  int ncu = 0;
  float *yhat = nullptr, *tgt = nullptr, *head_acc = nullptr, *terrain = nullptr,
        *params_in = nullptr;
  // resident training set
  float *data_terrain = nullptr, *data_params = nullptr, *data_tgt = nullptr;
  int data_n = 0;
  long adam_t = 0;
  double train_ms = 0, flops_per_sample = 0;
  uint64_t samples_trained = 0;
};

namespace {

int check_launch_u() {
  FS_HIP_TRY(hipGetLastError());
  return FS_OK;
}

int grid_for(long n) { return static_cast<int>(std::min<long>((n + 255) / 256, 4096)); }

int alloc_tensor(fs_unet *u, Tensor &t, int C, int level) {
  t.C = C;
  t.level = level;
  const size_t n = static_cast<size_t>(u->max_batch) * (u->H >> level) * (u->W >> level) * C;
  return fs::dev_alloc(&t.d, n);
}

long pixels(const fs_unet *u, int level, int B) {
  return static_cast<long>(B) * (u->H >> level) * (u->W >> level);
}

ConvSrc src_of(const Tensor &t) { return ConvSrc{t.d, nullptr, t.C, 0, 0}; }
// [lo upsampled, skip]
ConvSrc src_of(const Tensor &lo, const Tensor &skip) {
  return ConvSrc{lo.d, skip.d, lo.C, skip.C, 1};
}
ConvDst dst_of(const Tensor &t) {
  return ConvDst{t.d, nullptr, nullptr, nullptr, nullptr, 0};
}

template <int R>
int launch_conv_rows(fs_unet *u, const ConvSrc &src, const uint16_t *wt, const float *bias,
                     const ConvDst &dst, int nout, int Hl, int Wl, int relu, int B) {
  const int tx = (Wl + 15) / 16, ty = (Hl + R - 1) / R, tiles = tx * ty * B;
  const int groups = (tiles + kWaves - 1) / kWaves, nblk = nout / kNB;
  // two workgroups per CU in all; no more of them than groups to take
  const int per_xcd = std::max(1, std::min((groups + 7) / 8, 2 * u->ncu / 8 / nblk));
  hipLaunchKernelGGL(k_conv<R>, dim3(8 * nblk * per_xcd), dim3(64 * kWaves), 0, u->stream, src, wt,
                     bias, relu, dst, nout, Hl, Wl, tx, ty, tiles, groups);
  return check_launch_u();
}

// dst = conv3x3(src) with weights wt [tap][nout][cin].
int launch_conv(fs_unet *u, const ConvSrc &src, const uint16_t *wt, const float *bias,
                const ConvDst &dst, int nout, int Hl, int Wl, int relu, int B) {
  const int tx = (Wl + 15) / 16, ty = (Hl + 1) / 2, tiles = tx * ty * B;
  if (Hl < 8 || Wl < 16) {
    hipLaunchKernelGGL(k_conv_small<true>, dim3(tiles, nout / kNB), dim3(64), 0, u->stream, src, wt,
                       bias, relu, dst, nout, Hl, Wl, tx, ty, tiles);
    return check_launch_u();
  }
  // Up to a wave per CU, waves by themselves: a workgroup of k_conv would have
  // its four on one CU and wait for its weights in every step (one sample of 64
  // x 64 180 us, by themselves 160; of 128 x 128 174 and 167).  With two or four
  // waves per CU k_conv is level or ahead (four of 128 x 128: 198 against 204
  // and 229).
  if (static_cast<long>(tiles) * (nout / kNB) <= static_cast<long>(u->ncu)) {
    hipLaunchKernelGGL(k_conv_small<false>, dim3(tiles, nout / kNB), dim3(64), 0, u->stream, src,
                       wt, bias, relu, dst, nout, Hl, Wl, tx, ty, tiles);
    return check_launch_u();
  }
  // 8 rows a wave wherever that gives every SIMD a wave (1024 of them); below,
  // 2 rows: four of 128 x 128 take 198 us; 32 of 256 x 256 take as long with 4
  // rows as with 8
  const long waves = static_cast<long>((Wl + 15) / 16) * (Hl / 8) * B * (nout / kNB);
  if (waves >= 4l * u->ncu)
    return launch_conv_rows<8>(u, src, wt, bias, dst, nout, Hl, Wl, relu, B);
  return launch_conv_rows<2>(u, src, wt, bias, dst, nout, Hl, Wl, relu, B);
}

// conv + bias + ReLU into out; with pooled, also its 2 x 2 averages
int conv_fwd(fs_unet *u, const Conv &c, const ConvSrc &in, Tensor &out, const Tensor *pooled,
             int B) {
  ConvDst dst = dst_of(out);
  if (pooled) dst.pool = pooled->d;
  return launch_conv(u, in, c.wf, u->w + c.boff, dst, c.cout, u->H >> c.level, u->W >> c.level, 1,
                     B);
}

// Work split of the nine-tap weight-gradient kernel: about kDwTargetGroups
// workgroups per layer, the two that fit on every CU (1024 of them: 4.47 ms
// against 4.29 for the loss and gradients of 32 samples).  Levels whose size is
// not a multiple of the strips use k_conv3x3_dw.
constexpr long kDwTargetGroups = 512;
struct DwPlan {
  bool tiled = false;
  int nc = 0, ci_blocks = 0, blocks = 0, upc = 0, nchunks = 0;
  long strips = 0, units = 0, max_chunks = 0;
};
DwPlan dw_plan(int cout, int cin, int Hl, int Wl, int B) {
  DwPlan p;
  p.tiled = Hl % 8 == 0 && Wl % 16 == 0 && cin % 8 == 0 && cout % 32 == 0;
  if (!p.tiled) return p;
  p.nc = cout % 64 == 0 ? 2 : 1;
  const int rows = p.nc == 2 ? DwShape<2, 1>::R : DwShape<1, 2>::R;
  const int per_unit = p.nc == 2 ? DwShape<2, 1>::kStrips : DwShape<1, 2>::kStrips;
  p.ci_blocks = (cin + 31) / 32;
  p.blocks = cout / (32 * p.nc) * p.ci_blocks;
  p.strips = static_cast<long>(B) * (Hl / rows) * (Wl / 16);
  p.units = (p.strips + per_unit - 1) / per_unit;
  const long want = (kDwTargetGroups + p.blocks - 1) / p.blocks;
  p.max_chunks = std::min(want, p.units);
  p.upc = static_cast<int>((p.units + p.max_chunks - 1) / p.max_chunks);
  p.nchunks = static_cast<int>((p.units + p.upc - 1) / p.upc);
  return p;
}

// Pixels per chunk of the per-tap kernel, in whole 32s: up to 64 chunks, a few more
// where rounding the chunk down leaves a rest.  The number of chunks therefore
// does not always grow with the batch (352 x 352, level 2: 64 for 32 samples, 65 for
// 22).
struct TapChunks {
  long chunk;
  int n;
};
TapChunks tap_chunks(long M) {
  const long chunk = std::max<long>(2048, (M + 63) / 64 / 32 * 32);
  return {chunk, static_cast<int>((M + chunk - 1) / chunk)};
}

// Partial sums that the weight gradient of one layer needs for any batch up to
// max_batch.
size_t part_need(const Conv &c, int Hl, int Wl, int max_batch) {
  const DwPlan dp = dw_plan(c.cout, c.cin, Hl, Wl, max_batch);
  long chunks = dp.max_chunks;   // grows with the batch
  for (int B = 1; !dp.tiled && B <= max_batch; B++)
    chunks = std::max<long>(chunks, tap_chunks(static_cast<long>(B) * Hl * Wl).n);
  return static_cast<size_t>(chunks) * 9 * c.cout * c.cin;
}

// Gradients of one conv layer from gz, the gradient of its output before the
// ReLU: weight and bias gradients, and the input gradient into gin (if given).
int conv_bwd(fs_unet *u, const Conv &c, const ConvSrc &in, const Tensor &gz, const ConvDst *gin,
             int B) {
  const int Hl = u->H >> c.level, Wl = u->W >> c.level;
  const long M = pixels(u, c.level, B);
  // weight gradient, split over pixel chunks
  const size_t wn = 9ul * c.cout * c.cin;
  const DwPlan dp = dw_plan(c.cout, c.cin, Hl, Wl, B);
  if (dp.tiled) {
    if (static_cast<size_t>(dp.nchunks) * wn > u->part_n) return FS_ERR_INTERNAL;
    // the bias gradient is summed by the same kernel
    if (dp.nc == 2)
      hipLaunchKernelGGL((k_conv_dw<2, 1>), dim3(dp.blocks, dp.nchunks), dim3(kDwThreads), 0,
                         u->stream, gz.d, c.cout, in, u->part, u->g + c.boff, Hl, Wl, dp.strips,
                         dp.units, dp.upc, dp.ci_blocks);
    else
      hipLaunchKernelGGL((k_conv_dw<1, 2>), dim3(dp.blocks, dp.nchunks), dim3(kDwThreads), 0,
                         u->stream, gz.d, c.cout, in, u->part, u->g + c.boff, Hl, Wl, dp.strips,
                         dp.units, dp.upc, dp.ci_blocks);
    FS_TRY(check_launch_u());
    hipLaunchKernelGGL(k_reduce_chunks_wide, dim3(static_cast<unsigned>((wn + 63) / 64)),
                       dim3(1024), 0, u->stream, u->part, u->g + c.woff, static_cast<long>(wn),
                       dp.nchunks);
    FS_TRY(check_launch_u());
  } else {
    const TapChunks tc = tap_chunks(M);
    if (static_cast<size_t>(tc.n) * wn > u->part_n) return FS_ERR_INTERNAL;
    const int tiles = ((c.cout + 63) / 64) * ((c.cin + 63) / 64);
    hipLaunchKernelGGL(k_conv3x3_dw, dim3(tiles, 9, tc.n), dim3(256), 0, u->stream, gz.d,
                       c.cout, in, u->part, Hl, Wl, tc.chunk, M);
    FS_TRY(check_launch_u());
    hipLaunchKernelGGL(k_reduce_chunks, dim3(grid_for(static_cast<long>(wn))), dim3(256), 0,
                       u->stream, u->part, u->g + c.woff, static_cast<long>(wn), tc.n);
    FS_TRY(check_launch_u());
  }
  if (!dp.tiled) {
    const long bchunk = 4096;
    hipLaunchKernelGGL(k_bias_grad, dim3((M + bchunk - 1) / bchunk), dim3(256), 0, u->stream,
                       gz.d, c.cout, u->g + c.boff, M, bchunk);
    FS_TRY(check_launch_u());
  }
  if (gin) FS_TRY(launch_conv(u, src_of(gz), c.wb, nullptr, *gin, c.cin, Hl, Wl, 0, B));
  return FS_OK;
}

int pack_weights(fs_unet *u) {
  for (const Conv &c : u->conv) {
    hipLaunchKernelGGL(k_pack_weights, dim3(grid_for(9l * c.cout * c.cin)), dim3(256), 0,
                       u->stream, u->w + c.woff, c.wf, c.wb, c.cout, c.cin);
    FS_TRY(check_launch_u());
  }
  return FS_OK;
}

// conv layer indices: encoder 2L, 2L+1 (L = 0..3); decoder 8 + 2j, 9 + 2j for
// levels 2, 1, 0 (j = 0, 1, 2)
int enc(int L, int k) { return 2 * L + k; }
int dec(int L, int k) { return 8 + 2 * (2 - L) + k; }

int forward(fs_unet *u, const float *terrain_d, const float *params_d, int B,
            bool shared_terrain = false) {
  const long HW = static_cast<long>(u->H) * u->W;
  hipLaunchKernelGGL(k_pack_input, dim3(grid_for(B * HW)), dim3(256), 0, u->stream, terrain_d,
                     params_d, u->x0.d, B, HW, shared_terrain ? 0l : HW);
  FS_TRY(check_launch_u());
  const Tensor *in = &u->x0;
  for (int L = 0; L < kLevels; L++) {
    const Tensor *pooled = L < kLevels - 1 ? &u->p[L] : nullptr;
    FS_TRY(conv_fwd(u, u->conv[enc(L, 0)], src_of(*in), u->e_a[L], nullptr, B));
    FS_TRY(conv_fwd(u, u->conv[enc(L, 1)], src_of(u->e_a[L]), u->e[L], pooled, B));
    in = pooled;
  }
  const Tensor *lo = &u->e[kLevels - 1];
  for (int L = kLevels - 2; L >= 0; L--) {
    FS_TRY(conv_fwd(u, u->conv[dec(L, 0)], src_of(*lo, u->e[L]), u->d_a[L], nullptr, B));
    FS_TRY(conv_fwd(u, u->conv[dec(L, 1)], src_of(u->d_a[L]), u->d[L], nullptr, B));
    lo = &u->d[L];
  }
  const long M = pixels(u, 0, B);
  hipLaunchKernelGGL(k_head, dim3(grid_for(M)), dim3(256), 0, u->stream, u->d[0].d,
                     u->w + u->head_w, u->w + u->head_b, u->yhat, M);
  return check_launch_u();
}

// The encoder's levels from here down, the decoder and the head hold 95% of the
// parameters, at the end of the vector, and their gradients are there before
// the two largest levels' are.
constexpr int kDeepLevel = 2;

// gradients of the loss mean((yhat - tgt)^2) w.r.t. every parameter into g; deep_done
// is recorded behind those from kDeepLevel's on;
// head_acc[0] receives the loss
int backward(fs_unet *u, int B, hipEvent_t deep_done = nullptr) {
  const long M = pixels(u, 0, B);
  // every gradient that is added up by atomics starts from zero
  hipLaunchKernelGGL(k_fill_f32, dim3(grid_for(static_cast<long>(u->nparam))), dim3(256), 0,
                     u->stream, u->g, static_cast<long>(u->nparam), 0.f);
  hipLaunchKernelGGL(k_fill_f32, dim3(1), dim3(256), 0, u->stream, u->head_acc, 1l, 0.f);
  hipLaunchKernelGGL(k_head_grad, dim3(std::min<long>((4 * M + 255) / 256, 2048)), dim3(256), 0,
                     u->stream, u->d[0].d, u->w + u->head_w, u->yhat, u->tgt, u->gd[0].d,
                     u->head_acc, u->g + u->head_w, M);
  FS_TRY(check_launch_u());
  // decoder, top level first; the gradient of the concatenated input goes to
  // the level below (summed over the upsampling) and to the skip connection
  for (int L = 0; L <= kLevels - 2; L++) {
    const bool deepest = L + 1 == kLevels - 1;
    const Tensor &lo = deepest ? u->e[L + 1] : u->d[L + 1];
    ConvDst ga = dst_of(u->gd_a[L]);
    ga.mask = u->d_a[L].d;
    FS_TRY(conv_bwd(u, u->conv[dec(L, 1)], src_of(u->d_a[L]), u->gd[L], &ga, B));
    ConvDst gu = dst_of(u->ge[L]);
    gu.lo = deepest ? u->ge[L + 1].d : u->gd[L + 1].d;
    gu.lo_mask = lo.d;
    gu.c1 = lo.C;
    FS_TRY(conv_bwd(u, u->conv[dec(L, 0)], src_of(lo, u->e[L]), u->gd_a[L], &gu, B));
  }
  // encoder, bottom level first; ge[L] holds the skip gradient, the pooled
  // path's gradient is added
  for (int L = kLevels - 1; L >= 0; L--) {
    if (L < kLevels - 1) {
      hipLaunchKernelGGL(k_pool_grad, dim3(grid_for(pixels(u, L, B) * u->ge[L].C / 8)),
                         dim3(256), 0, u->stream, u->gp[L].d, u->ge[L].d, u->e[L].d, B, u->H >> L,
                         u->W >> L, u->ge[L].C);
      FS_TRY(check_launch_u());
    }
    ConvDst ga = dst_of(u->ge_a[L]);
    ga.mask = u->e_a[L].d;
    FS_TRY(conv_bwd(u, u->conv[enc(L, 1)], src_of(u->e_a[L]), u->ge[L], &ga, B));
    const Tensor &in = L == 0 ? u->x0 : u->p[L - 1];
    const ConvDst gp = L == 0 ? ConvDst{} : dst_of(u->gp[L - 1]);
    FS_TRY(conv_bwd(u, u->conv[enc(L, 0)], src_of(in), u->ge_a[L], L == 0 ? nullptr : &gp, B));
    if (L == kDeepLevel && deep_done) FS_HIP_TRY(hipEventRecord(deep_done, u->stream));
  }
  return FS_OK;
}

void free_unet(fs_unet *u) {
  if (!u) return;
  (void)hipSetDevice(u->device);
  if (u->stream) (void)hipStreamSynchronize(u->stream);
  if (u->copy) (void)hipStreamSynchronize(u->copy);
  std::vector<void *> ptrs = {u->w, u->g, u->m, u->v, u->part, u->yhat, u->tgt, u->head_acc,
                              u->terrain, u->params_in, u->data_terrain, u->data_params,
                              u->data_tgt, u->x0.d};
  for (int L = 0; L < kLevels; L++) {
    ptrs.push_back(u->e_a[L].d);
    ptrs.push_back(u->e[L].d);
    ptrs.push_back(u->ge_a[L].d);
    ptrs.push_back(u->ge[L].d);
  }
  for (int L = 0; L < kLevels - 1; L++)
    for (Tensor *t : {&u->p[L], &u->d_a[L], &u->d[L], &u->gp[L], &u->gd_a[L], &u->gd[L]})
      ptrs.push_back(t->d);
  for (Conv &c : u->conv) {
    ptrs.push_back(c.wf);
    ptrs.push_back(c.wb);
  }
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  for (hipEvent_t e : u->copy_ev)
    if (e) (void)hipEventDestroy(e);
  if (u->copy) (void)hipStreamDestroy(u->copy);
  if (u->stream) (void)hipStreamDestroy(u->stream);
  delete u;
}

int check_unet(fs_unet *u) {
  if (!u) return FS_ERR_INVALID_ARGUMENT;
  FS_HIP_TRY(hipSetDevice(u->device));
  return FS_OK;
}

int upload_batch(fs_unet *u, const float *terrain, const float *params, const float *tgt,
                 int B) {
  const size_t HW = static_cast<size_t>(u->H) * u->W;
  FS_HIP_TRY(hipMemcpyAsync(u->terrain, terrain, B * HW * sizeof(float), hipMemcpyHostToDevice,
                            u->stream));
  FS_HIP_TRY(hipMemcpyAsync(u->params_in, params, B * 3 * sizeof(float), hipMemcpyHostToDevice,
                            u->stream));
  if (tgt)
    FS_HIP_TRY(hipMemcpyAsync(u->tgt, tgt, B * HW * sizeof(float), hipMemcpyHostToDevice,
                              u->stream));
  return FS_OK;
}

}  // namespace

extern "C" {

int fs_unet_create(int height, int width, int max_batch, uint64_t seed, int device,
                   fs_unet **out) {
  if (!out) return FS_ERR_INVALID_ARGUMENT;
  *out = nullptr;
  if (height < 32 || width < 32 || height % 32 || width % 32 || max_batch < 1 ||
      static_cast<long long>(height) * width * max_batch >= (1ll << 31))
    return FS_ERR_DIMENSIONS;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0 || device < 0 || device >= ndev) {
    fs::set_last_error("no HIP device " + std::to_string(device));
    return FS_ERR_NO_DEVICE;
  }
  fs_unet *u = new (std::nothrow) fs_unet();
  if (!u) return FS_ERR_OUT_OF_MEMORY;
  struct Guard {
    fs_unet *u;
    ~Guard() { if (u) free_unet(u); }
  } guard{u};
  u->H = height;
  u->W = width;
  u->max_batch = max_batch;
  u->device = device;
  FS_HIP_TRY(hipSetDevice(device));
  FS_HIP_TRY(hipStreamCreateWithFlags(&u->stream, hipStreamNonBlocking));
  FS_HIP_TRY(hipStreamCreateWithFlags(&u->copy, hipStreamNonBlocking));
  for (hipEvent_t &e : u->copy_ev) FS_HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  FS_HIP_TRY(hipDeviceGetAttribute(&u->ncu, hipDeviceAttributeMultiprocessorCount, device));
  // layers
  auto add = [&](int cin, int cout, int level) {
    Conv c;
    c.cin = cin;
    c.cout = cout;
    c.level = level;
    u->conv.push_back(c);
  };
  for (int L = 0; L < kLevels; L++) {
    add(L == 0 ? kInChannels : kWidth[L - 1], kWidth[L], L);
    add(kWidth[L], kWidth[L], L);
  }
  for (int L = kLevels - 2; L >= 0; L--) {
    const int below = L == kLevels - 2 ? kWidth[kLevels - 1] : kWidth[L + 1];
    add(below + kWidth[L], kWidth[L], L);
    add(kWidth[L], kWidth[L], L);
  }
  size_t off = 0;
  for (Conv &c : u->conv) {
    c.woff = off;
    off += 9ul * c.cout * c.cin;
    c.boff = off;
    off += c.cout;
  }
  u->head_w = off;
  off += kWidth[0];
  u->head_b = off;
  off += 1;
  u->nparam = off;
  // flops of one forward pass per sample: 2 per multiply-add
  double fl = 0;
  for (const Conv &c : u->conv)
    fl += 2.0 * 9 * c.cin * c.cout * (static_cast<double>(height >> c.level) * (width >> c.level));
  u->flops_per_sample = fl;

  FS_TRY(fs::dev_alloc(&u->w, off));
  FS_TRY(fs::dev_alloc(&u->g, off));
  FS_TRY(fs::dev_alloc(&u->m, off));
  FS_TRY(fs::dev_alloc(&u->v, off));
  for (Conv &c : u->conv) {
    FS_TRY(fs::dev_alloc(&c.wf, 9ul * c.cout * c.cin));
    FS_TRY(fs::dev_alloc(&c.wb, 9ul * c.cout * c.cin));
  }
  size_t part = 0;
  for (const Conv &c : u->conv)
    part = std::max(part, part_need(c, height >> c.level, width >> c.level, max_batch));
  u->part_n = part;
  FS_TRY(fs::dev_alloc(&u->part, part));
  FS_TRY(alloc_tensor(u, u->x0, kInChannels, 0));
  for (int L = 0; L < kLevels; L++) {
    FS_TRY(alloc_tensor(u, u->e_a[L], kWidth[L], L));
    FS_TRY(alloc_tensor(u, u->e[L], kWidth[L], L));
    FS_TRY(alloc_tensor(u, u->ge_a[L], kWidth[L], L));
    FS_TRY(alloc_tensor(u, u->ge[L], kWidth[L], L));
  }
  for (int L = 0; L < kLevels - 1; L++) {
    FS_TRY(alloc_tensor(u, u->p[L], kWidth[L], L + 1));
    FS_TRY(alloc_tensor(u, u->gp[L], kWidth[L], L + 1));
    FS_TRY(alloc_tensor(u, u->d_a[L], kWidth[L], L));
    FS_TRY(alloc_tensor(u, u->gd_a[L], kWidth[L], L));
    FS_TRY(alloc_tensor(u, u->d[L], kWidth[L], L));
    FS_TRY(alloc_tensor(u, u->gd[L], kWidth[L], L));
  }
  const size_t HWB = static_cast<size_t>(max_batch) * height * width;
  FS_TRY(fs::dev_alloc(&u->yhat, HWB));
  FS_TRY(fs::dev_alloc(&u->tgt, HWB));
  FS_TRY(fs::dev_alloc(&u->terrain, HWB));
  FS_TRY(fs::dev_alloc(&u->params_in, 3ul * max_batch));
  FS_TRY(fs::dev_alloc(&u->head_acc, 64));
  // He-normal initial weights, zero biases (host RNG, reproducible per seed)
  std::vector<float> w(off, 0.f);
  std::mt19937_64 rng(seed);
  for (const Conv &c : u->conv) {
    std::normal_distribution<float> nd(0.f, std::sqrt(2.0f / (9.0f * c.cin)));
    for (size_t i = 0; i < 9ul * c.cout * c.cin; i++) w[c.woff + i] = nd(rng);
  }
  {
    std::normal_distribution<float> nd(0.f, std::sqrt(1.0f / kWidth[0]));
    for (int i = 0; i < kWidth[0]; i++) w[u->head_w + i] = nd(rng);
  }
  FS_HIP_TRY(hipMemcpy(u->w, w.data(), off * sizeof(float), hipMemcpyHostToDevice));
  FS_HIP_TRY(hipMemset(u->m, 0, off * sizeof(float)));
  FS_HIP_TRY(hipMemset(u->v, 0, off * sizeof(float)));
  FS_HIP_TRY(hipMemset(u->g, 0, off * sizeof(float)));
  FS_TRY(pack_weights(u));
  FS_HIP_TRY(hipStreamSynchronize(u->stream));
  guard.u = nullptr;
  *out = u;
  return FS_OK;
}

int fs_unet_destroy(fs_unet *u) {
  if (!u) return FS_ERR_INVALID_ARGUMENT;
  free_unet(u);
  return FS_OK;
}

int fs_unet_param_count(fs_unet *u, size_t *n) {
  if (!u || !n) return FS_ERR_INVALID_ARGUMENT;
  *n = u->nparam;
  return FS_OK;
}

int fs_unet_get_params(fs_unet *u, float *p, size_t n) {
  FS_TRY(check_unet(u));
  if (!p) return FS_ERR_INVALID_ARGUMENT;
  if (n != u->nparam) return FS_ERR_BUFFER_SIZE;
  FS_HIP_TRY(hipStreamSynchronize(u->stream));
  FS_HIP_TRY(hipMemcpy(p, u->w, n * sizeof(float), hipMemcpyDeviceToHost));
  return FS_OK;
}

int fs_unet_set_params(fs_unet *u, const float *p, size_t n) {
  FS_TRY(check_unet(u));
  if (!p) return FS_ERR_INVALID_ARGUMENT;
  if (n != u->nparam) return FS_ERR_BUFFER_SIZE;
  FS_HIP_TRY(hipStreamSynchronize(u->stream));
  FS_HIP_TRY(hipMemcpy(u->w, p, n * sizeof(float), hipMemcpyHostToDevice));
  FS_TRY(pack_weights(u));
  FS_HIP_TRY(hipStreamSynchronize(u->stream));
  return FS_OK;
}

int fs_unet_layer_shapes(fs_unet *u, int *cin, int *cout, int *level, int capacity, int *count) {
  if (!u || !count) return FS_ERR_INVALID_ARGUMENT;
  *count = static_cast<int>(u->conv.size());
  if (!cin && !cout && !level) return FS_OK;
  if (capacity < *count) return FS_ERR_BUFFER_SIZE;
  for (int i = 0; i < *count; i++) {
    if (cin) cin[i] = u->conv[i].cin;
    if (cout) cout[i] = u->conv[i].cout;
    if (level) level[i] = u->conv[i].level;
  }
  return FS_OK;
}

int fs_unet_forward(fs_unet *u, const float *terrain, const float *params, int batch, float *y) {
  FS_TRY(check_unet(u));
  if (!terrain || !params || !y) return FS_ERR_INVALID_ARGUMENT;
  const size_t HW = static_cast<size_t>(u->H) * u->W;
  for (int b0 = 0; b0 < batch; b0 += u->max_batch) {
    const int B = std::min(u->max_batch, batch - b0);
    FS_TRY(upload_batch(u, terrain + b0 * HW, params + 3ul * b0, nullptr, B));
    FS_TRY(forward(u, u->terrain, u->params_in, B));
    FS_HIP_TRY(hipMemcpyAsync(y + b0 * HW, u->yhat, B * HW * sizeof(float),
                              hipMemcpyDeviceToHost, u->stream));
  }
  FS_HIP_TRY(hipStreamSynchronize(u->stream));
  return FS_OK;
}

int fs_unet_loss_grad(fs_unet *u, const float *terrain, const float *params, const float *tgt,
                      int batch, float *loss, float *grad, size_t n) {
  FS_TRY(check_unet(u));
  if (!terrain || !params || !tgt || !loss) return FS_ERR_INVALID_ARGUMENT;
  if (batch < 1 || batch > u->max_batch) return FS_ERR_INVALID_ARGUMENT;
  if (grad && n != u->nparam) return FS_ERR_BUFFER_SIZE;
  // The host's copies run beside the kernels (8 MB of targets and 5.5 MB of
  // gradients for 32 samples of 256 x 256: 4.08 ms one after the other, now
  // 3.55): the targets' while the forward pass, which does not read them, runs,
  // most of the gradients' during the last layers' backward pass.
  const size_t npix = static_cast<size_t>(batch) * u->H * u->W;
  const size_t head = grad ? u->conv[enc(kDeepLevel, 0)].woff : 0;
  int st = [&] {
    FS_HIP_TRY(hipEventRecord(u->copy_ev[0], u->stream));
    FS_TRY(upload_batch(u, terrain, params, nullptr, batch));
    FS_TRY(forward(u, u->terrain, u->params_in, batch));
    FS_HIP_TRY(hipStreamWaitEvent(u->copy, u->copy_ev[0], 0));
    FS_HIP_TRY(hipMemcpyAsync(u->tgt, tgt, npix * sizeof(float), hipMemcpyHostToDevice, u->copy));
    FS_HIP_TRY(hipEventRecord(u->copy_ev[1], u->copy));
    FS_HIP_TRY(hipStreamWaitEvent(u->stream, u->copy_ev[1], 0));
    FS_TRY(backward(u, batch, u->copy_ev[0]));
    if (grad) {
      FS_HIP_TRY(hipStreamWaitEvent(u->copy, u->copy_ev[0], 0));
      FS_HIP_TRY(hipMemcpyAsync(grad + head, u->g + head, (n - head) * sizeof(float),
                                hipMemcpyDeviceToHost, u->copy));
      FS_HIP_TRY(hipMemcpyAsync(grad, u->g, head * sizeof(float), hipMemcpyDeviceToHost,
                                u->stream));
    }
    FS_HIP_TRY(hipMemcpyAsync(loss, u->head_acc, sizeof(float), hipMemcpyDeviceToHost, u->stream));
    return FS_OK;
  }();
  // the caller's arrays are free again, whatever happened: both streams are
  // waited for, and the first failure is reported
  for (hipStream_t s : {u->copy, u->stream}) {
    const int waited = [&] {
      FS_HIP_TRY(hipStreamSynchronize(s));
      return FS_OK;
    }();
    if (st == FS_OK) st = waited;
  }
  return st;
}

int fs_unet_set_data(fs_unet *u, const float *terrain, const float *params, const float *tgt,
                     int count) {
  FS_TRY(check_unet(u));
  if (!terrain || !params || !tgt || count < 1) return FS_ERR_INVALID_ARGUMENT;
  const size_t HW = static_cast<size_t>(u->H) * u->W;
  FS_HIP_TRY(hipStreamSynchronize(u->stream));
  for (float *p : {u->data_terrain, u->data_params, u->data_tgt})
    if (p) (void)hipFree(p);
  u->data_terrain = u->data_params = u->data_tgt = nullptr;
  u->data_n = 0;
  FS_TRY(fs::dev_alloc(&u->data_terrain, count * HW));
  FS_TRY(fs::dev_alloc(&u->data_params, 3ul * count));
  FS_TRY(fs::dev_alloc(&u->data_tgt, count * HW));
  FS_HIP_TRY(hipMemcpy(u->data_terrain, terrain, count * HW * sizeof(float), hipMemcpyHostToDevice));
  FS_HIP_TRY(hipMemcpy(u->data_params, params, 3ul * count * sizeof(float), hipMemcpyHostToDevice));
  FS_HIP_TRY(hipMemcpy(u->data_tgt, tgt, count * HW * sizeof(float), hipMemcpyHostToDevice));
  u->data_n = count;
  return FS_OK;
}

int fs_unet_train(fs_unet *u, int epochs, int batch, float lr, uint64_t seed, float *epoch_loss) {
  FS_TRY(check_unet(u));
  if (epochs < 1 || batch < 1 || batch > u->max_batch || !(lr > 0)) return FS_ERR_INVALID_ARGUMENT;
  if (u->data_n < batch) return FS_ERR_INVALID_ARGUMENT;
  const size_t HW = static_cast<size_t>(u->H) * u->W;
  const int per_epoch = u->data_n / batch;
  const long total = static_cast<long>(epochs) * per_epoch;
  std::mt19937_64 rng(seed);
  std::vector<int> order(u->data_n);
  for (int i = 0; i < u->data_n; i++) order[i] = i;
  std::vector<float> losses(per_epoch);
  float *loss_d = nullptr;
  FS_TRY(fs::dev_alloc(&loss_d, static_cast<size_t>(per_epoch)));
  struct Free {
    float *p;
    ~Free() { if (p) (void)hipFree(p); }
  } fr{loss_d};
  const auto t0 = std::chrono::steady_clock::now();
  long step = 0;
  for (int ep = 0; ep < epochs; ep++) {
    std::shuffle(order.begin(), order.end(), rng);
    for (int s = 0; s < per_epoch; s++, step++) {
      // gather the minibatch device-to-device
      for (int b = 0; b < batch; b++) {
        const int i = order[s * batch + b];
        FS_HIP_TRY(hipMemcpyAsync(u->terrain + b * HW, u->data_terrain + i * HW, HW * sizeof(float),
                                  hipMemcpyDeviceToDevice, u->stream));
        FS_HIP_TRY(hipMemcpyAsync(u->tgt + b * HW, u->data_tgt + i * HW, HW * sizeof(float),
                                  hipMemcpyDeviceToDevice, u->stream));
        FS_HIP_TRY(hipMemcpyAsync(u->params_in + 3 * b, u->data_params + 3l * i,
                                  3 * sizeof(float), hipMemcpyDeviceToDevice, u->stream));
      }
      FS_TRY(forward(u, u->terrain, u->params_in, batch));
      FS_TRY(backward(u, batch));
      FS_HIP_TRY(hipMemcpyAsync(loss_d + s, u->head_acc, sizeof(float), hipMemcpyDeviceToDevice,
                                u->stream));
      // cosine learning-rate decay to lr/20
      const double frac = total > 1 ? static_cast<double>(step) / (total - 1) : 1.0;
      const float lr_t = static_cast<float>(lr * (0.05 + 0.95 * 0.5 * (1.0 + std::cos(M_PI * frac))));
      u->adam_t++;
      const float c1 = 1.f - std::pow(0.9f, static_cast<float>(u->adam_t));
      const float c2 = 1.f - std::pow(0.999f, static_cast<float>(u->adam_t));
      hipLaunchKernelGGL(k_adam, dim3(grid_for(static_cast<long>(u->nparam))), dim3(256), 0,
                         u->stream, u->w, u->g, u->m, u->v, static_cast<long>(u->nparam), lr_t,
                         0.9f, 0.999f, 1e-8f, c1, c2);
      FS_TRY(check_launch_u());
      FS_TRY(pack_weights(u));
    }
    FS_HIP_TRY(hipMemcpyAsync(losses.data(), loss_d, per_epoch * sizeof(float),
                              hipMemcpyDeviceToHost, u->stream));
    FS_HIP_TRY(hipStreamSynchronize(u->stream));
    double s = 0;
    for (float l : losses) s += l;
    if (epoch_loss) epoch_loss[ep] = static_cast<float>(s / per_epoch);
  }
  u->train_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  u->samples_trained += static_cast<uint64_t>(total) * batch;
  return FS_OK;
}

int fs_unet_rank(fs_unet *u, const float *terrain, const float *params, int count,
                 const float *target, float *misfit) {
  FS_TRY(check_unet(u));
  if (!terrain || !params || !target || !misfit || count < 1) return FS_ERR_INVALID_ARGUMENT;
  const size_t HW = static_cast<size_t>(u->H) * u->W;
  float *p_d = nullptr, *sq_d = nullptr;
  FS_TRY(fs::dev_alloc(&p_d, 3ul * count));
  struct Free {
    float *a, *b;
    ~Free() {
      if (a) (void)hipFree(a);
      if (b) (void)hipFree(b);
    }
  } fr{p_d, nullptr};
  FS_TRY(fs::dev_alloc(&sq_d, static_cast<size_t>(count)));
  fr.b = sq_d;
  FS_HIP_TRY(hipMemcpyAsync(p_d, params, 3ul * count * sizeof(float), hipMemcpyHostToDevice,
                            u->stream));
  // terrain in u->terrain[0], target in u->tgt[0]
  FS_HIP_TRY(hipMemcpyAsync(u->terrain, terrain, HW * sizeof(float), hipMemcpyHostToDevice,
                            u->stream));
  FS_HIP_TRY(hipMemcpyAsync(u->tgt, target, HW * sizeof(float), hipMemcpyHostToDevice, u->stream));
  hipLaunchKernelGGL(k_fill_f32, dim3(grid_for(count)), dim3(256), 0, u->stream, sq_d,
                     static_cast<long>(count), 0.f);
  for (int b0 = 0; b0 < count; b0 += u->max_batch) {
    const int B = std::min(u->max_batch, count - b0);
    FS_TRY(forward(u, u->terrain, p_d + 3l * b0, B, true));
    hipLaunchKernelGGL(k_sq_misfit, dim3(static_cast<unsigned>(std::min<size_t>((HW + 255) / 256, 64)), B),
                       dim3(256), 0, u->stream, u->yhat, u->tgt, sq_d + b0, u->H, u->W);
    FS_TRY(check_launch_u());
  }
  std::vector<float> sq(count);
  FS_HIP_TRY(hipMemcpyAsync(sq.data(), sq_d, count * sizeof(float), hipMemcpyDeviceToHost,
                            u->stream));
  FS_HIP_TRY(hipStreamSynchronize(u->stream));
  const double ninterior = static_cast<double>(u->H - 4) * (u->W - 4);
  for (int i = 0; i < count; i++) misfit[i] = static_cast<float>(std::sqrt(sq[i] / ninterior));
  return FS_OK;
}

int fs_unet_stats(fs_unet *u, double *train_ms, double *flops_per_sample, uint64_t *samples) {
  if (!u) return FS_ERR_INVALID_ARGUMENT;
  if (train_ms) *train_ms = u->train_ms;
  if (flops_per_sample) *flops_per_sample = u->flops_per_sample;
  if (samples) *samples = u->samples_trained;
  return FS_OK;
}

}  // extern "C"
