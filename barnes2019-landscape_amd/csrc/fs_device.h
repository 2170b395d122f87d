// fs_device.h -- device code of the FastScape library: constants, lane and
// wave helpers, and every kernel.  Included by each HIP translation unit of
// the library; everything here has internal linkage.
#ifndef FS_DEVICE_H
#define FS_DEVICE_H

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstddef>
#include <cstdint>

#include "fastscape.h"
#include "fs_internal.h"
#include "fs_receiver.h"

namespace {

constexpr int kWave = 64;
constexpr uint8_t kNoFlow = 0xFF;
constexpr int kWalkCap = 64;           // hops walked per cell in k_topology
constexpr int kJumpPasses = 12;        // kWalkCap * 2^10 > FS_MAX_LEVELS
constexpr int kScanBlock = 256;
constexpr int kRootItems = 16;         // cells per thread in k_roots
constexpr int kRootTile = kScanBlock * kRootItems;
constexpr int kBfsItems = 8;           // stack entries per thread in k_bfs
constexpr int kBfsTile = kScanBlock * kBfsItems;
constexpr int kSmallBlock = 1024;
constexpr int kSmallItems = 4;
constexpr int kSmallLevel = kSmallBlock * kSmallItems;  // one-workgroup levels
constexpr int kNewtonCap = 100;
// Tile-path steps are launched in batches of up to kMaxBatch without a host
// round trip; each step reports into a slot of its own.
constexpr int kMaxBatch = 32;
constexpr int kSlotOver = 0;           // tiles deeper than the halo: the step was not taken
constexpr int kSlotDeepest = 1;        // deepest level (32-cell halo)
constexpr int kSlotStop = 2;           // the step was not reached
constexpr int kSlotInts = 4;
constexpr int kHdrSlots = 4;
// header: maxdepth, n_unfinished, err, spare; the batch's slots
constexpr int kHdrInts = kHdrSlots + kMaxBatch * kSlotInts;
constexpr int kHdrCounts = 1024;       // level counts fetched with the header
// After the level counts: one "cells still unfinished" flag per pointer-
// jumping pass, so the passes after the last needed one return at once.
constexpr int kHdrJump = kHdrInts + FS_MAX_LEVELS + 3;
constexpr int kHdrAlloc = kHdrJump + kJumpPasses + 1;   // header ints allocated
constexpr int kTopoBlocks = 2048;
constexpr int kJumpBlocks = 1024;
constexpr int kJumpHist = 2048;         // levels k_jump counts in LDS

// device error bits (hdr[2])
constexpr int kErrLookback = 1, kErrNewton = 2, kErrIndex = 4, kErrDepth = 8;

// ---------------------------------------------------------------------------
// neighbourhood encodings
// ---------------------------------------------------------------------------
// Receiver direction r = 0..7 is W, NW, N, NE, E, SE, S, SW (RB:79-82); its
// offset is nshift[r] = {-1, -W-1, -W, -W+1, 1, W+1, W, W-1} (RB:137).
__device__ __forceinline__ int dir_offset(int r, int W) {
  constexpr unsigned kDx = (0u << 0) | (0u << 2) | (1u << 4) | (2u << 6) |
                           (2u << 8) | (2u << 10) | (1u << 12) | (0u << 14);
  constexpr unsigned kDy = (1u << 0) | (0u << 2) | (0u << 4) | (0u << 6) |
                           (1u << 8) | (2u << 10) | (2u << 12) | (2u << 14);
  const int dx = static_cast<int>((kDx >> (2 * r)) & 3u) - 1;
  const int dy = static_cast<int>((kDy >> (2 * r)) & 3u) - 1;
  return dy * W + dx;
}

// Donor bitmask slot j = 0..7 is the neighbour at offset
// {-W-1, -W, -W+1, -1, +1, W-1, W, W+1}[j]: ascending cell index, so the set
// bits in slot order list the donors in the order RB's push builds them
// (RB:194-202).  The neighbour in slot j is a donor iff its receiver
// direction is kSlotDir[j].
__device__ __forceinline__ int slot_offset(int j, int W) {
  constexpr unsigned kSx = (0u << 0) | (1u << 2) | (2u << 4) | (0u << 6) |
                           (2u << 8) | (0u << 10) | (1u << 12) | (2u << 14);
  constexpr unsigned kSy = (0u << 0) | (0u << 2) | (0u << 4) | (1u << 6) |
                           (1u << 8) | (2u << 10) | (2u << 12) | (2u << 14);
  const int dx = static_cast<int>((kSx >> (2 * j)) & 3u) - 1;
  const int dy = static_cast<int>((kSy >> (2 * j)) & 3u) - 1;
  return dy * W + dx;
}

// ---------------------------------------------------------------------------
// scans
// ---------------------------------------------------------------------------
// Exclusive prefix sum over the block; *total gets the block sum.  sh holds
// BLOCK/64 + 1 words.  Ends with a barrier, so sh may be reused at once.
template <int BLOCK>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *total,
                                                    uint32_t *sh) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  uint32_t x = v;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == kWave - 1) sh[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t run = 0;
    for (int w = 0; w < BLOCK / kWave; w++) {
      const uint32_t t = sh[w];
      sh[w] = run;
      run += t;
    }
    sh[BLOCK / kWave] = run;
  }
  __syncthreads();
  const uint32_t ex = sh[wid] + x - v;
  *total = sh[BLOCK / kWave];
  __syncthreads();
  return ex;
}

// Tile status word: [epoch:30 | flag:2 | value:32].  flag 1 = tile aggregate,
// 2 = inclusive prefix.  A word whose epoch is not the launch's epoch is
// "not yet published", so the array never needs clearing.
__device__ __forceinline__ uint64_t status_word(uint32_t epoch, uint32_t flag, uint32_t v) {
  return (static_cast<uint64_t>(epoch & 0x3fffffffu) << 34) |
         (static_cast<uint64_t>(flag) << 32) | v;
}

// Decoupled look-back (Merrill & Garland, "Single-pass Parallel Prefix Scan
// with Decoupled Look-back", 2016), run by one full wave.  Publishes the
// tile's aggregate, sums predecessors' aggregates 64 at a time until an
// inclusive prefix is found, publishes its own inclusive prefix and returns
// the tile's exclusive prefix in every lane.  Tiles are numbered by an atomic
// ticket, so every predecessor is resident and publishes its aggregate
// without waiting; the wait is still bounded and reported in *err.
__device__ uint32_t lookback(uint64_t *status, uint32_t tile, uint32_t epoch,
                             uint32_t agg, int32_t *err) {
  const int lane = threadIdx.x & (kWave - 1);
  epoch &= 0x3fffffffu;
  if (tile == 0) {
    if (lane == 0)
      __hip_atomic_store(&status[0], status_word(epoch, 2, agg), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    return 0;
  }
  if (lane == 0)
    __hip_atomic_store(&status[tile], status_word(epoch, 1, agg), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  uint32_t excl = 0;
  long long base = static_cast<long long>(tile) - 1;
  int spins = 0;
  while (true) {
    const long long idx = base - lane;
    uint64_t w = status_word(epoch, 2, 0);
    if (idx >= 0)
      w = __hip_atomic_load(&status[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t flag = static_cast<uint32_t>(w >> 32) & 3u;
    const bool valid = (static_cast<uint32_t>(w >> 34) == epoch) && flag != 0;
    const unsigned long long inval = __ballot(!valid);
    const unsigned long long pmask = __ballot(valid && flag == 2);
    const int first_p = pmask ? __builtin_ctzll(pmask) : kWave;
    const int first_inv = inval ? __builtin_ctzll(inval) : kWave;
    if (first_inv < first_p) {
      if (++spins > (1 << 22)) {
        if (lane == 0) atomicOr(err, kErrLookback);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    uint32_t v = (lane <= first_p) ? static_cast<uint32_t>(w) : 0u;
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    excl += v;
    if (first_p < kWave) break;
    base -= kWave;
  }
  if (lane == 0)
    __hip_atomic_store(&status[tile], status_word(epoch, 2, excl + agg),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return excl;
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
// Opens a slot for another attempt of its step.
__global__ void k_slot_reset(int32_t *slot) {
  if (threadIdx.x < kSlotInts) slot[threadIdx.x] = 0;
}

__global__ void k_fill_counts(int32_t *hdr, int n_counts) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    hdr[0] = 0;   // maxdepth
    hdr[1] = 0;   // n_unfinished
  }
  if (i < n_counts) hdr[kHdrInts + i] = 0;
  if (i <= kJumpPasses) hdr[kHdrJump + i] = 0;
}

// ComputeReceivers (RB:160-182).  fs::receiver_fast picks the reference's
// direction -- steepest (hc - h[n]) / dr[n] over n = 0..7 with a strict '>'
// from 0, ties to the lowest n, flat cells and pits NO_FLOW -- and divides only
// in the rare cells that need it (near-ties, extreme magnitudes).  Rows are
// read through buffer resources built per row in scalar registers: the lane's
// column is a constant offset, so no vector instructions go to addresses.
constexpr int kRsrcWord3 = 0x00020000;          // raw (unformatted) buffer, gfx9
using v4u = unsigned __attribute__((ext_vector_type(4)));
using v2u = unsigned __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const void *row, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(row), 0, static_cast<int>(bytes),
                                           kRsrcWord3);
}

// columns x-1, x, x+1 of a row; xo = 8*(x-1) (a row of W doubles is below
// 2^32 bytes: W*H < 2^31 with H >= 5)
__device__ __forceinline__ void load_cols(__amdgpu_buffer_rsrc_t r, uint32_t xo, double &l,
                                          double &c, double &rr) {
  const v4u a = __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(xo), 0, 0);
  const v2u b = __builtin_amdgcn_raw_buffer_load_b64(r, static_cast<int>(xo) + 16, 0, 0);
  l = __builtin_bit_cast(double, v2u{a.x, a.y});
  c = __builtin_bit_cast(double, v2u{a.z, a.w});
  rr = __builtin_bit_cast(double, b);
}

// Receivers of one grid: each wave owns 64 columns x kRecvShort rows, with all
// its kRecvShort + 2 rows requested before the first is used, so a cell waits
// for memory once.  A rolling window (32 rows per thread, one row ahead)
// left small grids to a chain of 32 dependent row loads on a few
// waves: 15 us at 101^2 and at 1000^2 alike.  Six rows were the best of 1 to
// 16 at every size: 19.1 -> 9.0 us at 1000^2, 22.4 -> 15.9 at 2048^2, 93.5 ->
// 86.3 at 6000^2, 227 -> 223.5 at 10000^2 (HIP events, their own 4 us
// included); four rows read 1.5 rows per row decided (241 us at 10000^2),
// sixteen leave too few waves (12.1 at 1000^2).  Bound by memory at the
// largest sizes (1.23 GB in 0.22 ms, a copy's rate; VALU active 71% of the cycles).
// On the tile path it also opens its step's slot.  prev is the slot of the
// batch's previous step (null for its first): when that step was not taken, a
// solve failed, or its drainage was no deeper than `shallow` levels (the
// smaller halo fits again; -1: no such limit), this step is not taken either,
// and nothing is written but the slot.
constexpr int kRecvShort = 6;
constexpr int kRecvGroups = 256 / kWave;   // row groups per workgroup
struct ShortRows {
  double l[kRecvShort + 2], c[kRecvShort + 2], r[kRecvShort + 2];
};
// Requests the rows of row group `group` in column x (past the grid's last
// row: that row again).
__device__ __forceinline__ void load_short(ShortRows &v, const double *__restrict__ h, int W, int H,
                                           int x, int group) {
  const uint32_t rowb = static_cast<uint32_t>(W) * 8u;
  const uint32_t xo = static_cast<uint32_t>(x - 1) * 8u;
  const int y0 = group * kRecvShort + 2;
#pragma unroll
  for (int k = 0; k < kRecvShort + 2; k++)
    load_cols(row_rsrc(h + static_cast<size_t>(min(y0 - 1 + k, H - 1)) * W, rowb), xo, v.l[k],
              v.c[k], v.r[k]);
}
__device__ __forceinline__ void decide_short(const ShortRows &v, uint8_t *__restrict__ rcv, int W,
                                             int H, int x, int group, double d_card,
                                             double d_diag) {
  const bool div_ok = fs::divisors_in_range(d_card, d_diag);
  const int y0 = group * kRecvShort + 2;
#pragma unroll
  for (int k = 0; k < kRecvShort; k++) {
    if (y0 + k >= H - 2) break;
    const double nb[8] = {v.l[k + 1], v.l[k],     v.c[k],     v.r[k],
                          v.r[k + 1], v.r[k + 2], v.c[k + 2], v.l[k + 2]};
    rcv[static_cast<size_t>(y0 + k) * W + x] =
        static_cast<uint8_t>(fs::receiver_fast(v.c[k + 1], nb, d_card, d_diag, div_ok));
  }
}

__global__ __launch_bounds__(256) void k_receivers(const double *__restrict__ h,
                                                   uint8_t *__restrict__ rcv, int W, int H,
                                                   double d_card, double d_diag,
                                                   const int32_t *__restrict__ hdr,
                                                   const int32_t *prev, int32_t *slot,
                                                   int shallow) {
  const int x = blockIdx.x * kWave + static_cast<int>(threadIdx.x % kWave) + 2;
  const int group = __builtin_amdgcn_readfirstlane(
      (blockIdx.z * gridDim.y + blockIdx.y) * kRecvGroups + threadIdx.x / kWave);
  if (x >= W - 2 || group * kRecvShort + 2 >= H - 2) return;
  ShortRows v;
  load_short(v, h, W, H, x, group);
  const bool stop = prev != nullptr && (prev[kSlotOver] != 0 || prev[kSlotStop] != 0 ||
                                        hdr[2] != 0 || prev[kSlotDeepest] <= shallow);
  if (slot != nullptr && x == 2 && group == 0) {   // one thread of the grid
    slot[kSlotOver] = 0;
    slot[kSlotDeepest] = 0;
    slot[kSlotStop] = stop ? 1 : 0;
  }
  if (stop) return;
  decide_short(v, rcv, W, H, x, group, d_card, d_diag);
}

// Donor bitmask and level of every cell.  Rows are strided over the grid so
// each block folds its level histogram in LDS before touching HBM.  The
// level is found by walking receivers (all reads hit L1/L2: the receiver
// field is one byte per cell and the walk moves one cell per hop); walks
// longer than kWalkCap hops record (cell reached, hops) for k_jump.
__global__ __launch_bounds__(256) void k_topology(
    const uint8_t *__restrict__ rcv, uint8_t *__restrict__ dmask,
    uint16_t *__restrict__ depth, unsigned long long *__restrict__ jump,
    int32_t *__restrict__ list, int32_t *__restrict__ hdr, int W, int H) {
  __shared__ int hist[kWalkCap + 1];
  __shared__ int smax;
  for (int i = threadIdx.x; i <= kWalkCap; i += blockDim.x) hist[i] = 0;
  if (threadIdx.x == 0) smax = 0;
  __syncthreads();
  int32_t *counts = hdr + kHdrInts;
  int local_max = 0;
  for (int y = blockIdx.x; y < H; y += gridDim.x) {
    const bool yin = y > 0 && y < H - 1;
    for (int x = threadIdx.x; x < W; x += blockDim.x) {
      const int c = y * W + x;
      uint32_t m = 0;
      if (yin && x > 0 && x < W - 1) {
        const uint8_t *up = rcv + c - W;
        const uint8_t *dn = rcv + c + W;
        m |= (up[-1] == 5) ? 0x01u : 0u;
        m |= (up[0] == 6) ? 0x02u : 0u;
        m |= (up[1] == 7) ? 0x04u : 0u;
        m |= (rcv[c - 1] == 4) ? 0x08u : 0u;
        m |= (rcv[c + 1] == 0) ? 0x10u : 0u;
        m |= (dn[-1] == 3) ? 0x20u : 0u;
        m |= (dn[0] == 2) ? 0x40u : 0u;
        m |= (dn[1] == 1) ? 0x80u : 0u;
      }
      dmask[c] = static_cast<uint8_t>(m);
      int cur = c, d = 0;
      int r = rcv[c];
      while (r < 8 && d < kWalkCap) {
        cur += dir_offset(r, W);
        d++;
        r = rcv[cur];
      }
      if (r >= 8) {
        depth[c] = static_cast<uint16_t>(d);
        atomicAdd(&hist[d], 1);
        local_max = max(local_max, d);
      } else {
        depth[c] = 0xFFFF;
        jump[c] = (static_cast<unsigned long long>(d) << 32) | static_cast<uint32_t>(cur);
        const int slot = atomicAdd(&hdr[1], 1);
        list[slot] = c;
      }
    }
  }
  atomicMax(&smax, local_max);
  __syncthreads();
  for (int i = threadIdx.x; i <= kWalkCap; i += blockDim.x)
    if (hist[i]) atomicAdd(&counts[i], hist[i]);
  if (threadIdx.x == 0) atomicMax(&hdr[0], smax);
}

// One pointer-jumping pass over the cells k_topology left unfinished: a cell
// whose recorded ancestor has a level takes level = hops + that level;
// otherwise it jumps to its ancestor's ancestor.  (ancestor, hops) pairs are
// read and written as one 64-bit word, so every pair a thread sees is
// consistent and the update is safe in place.  A pass that leaves a cell
// unfinished raises the next pass's flag; a pass whose flag is down (the
// previous pass finished every cell) returns at once.
__global__ __launch_bounds__(256) void k_jump(const int32_t *__restrict__ list,
                                              uint16_t *depth, unsigned long long *jump,
                                              int32_t *hdr, int pass) {
  // level counts below kJumpHist and the deepest level are folded per block
  // in LDS: finished cells share a few hundred levels, so global atomics per
  // cell would queue on the same words
  __shared__ int hist[kJumpHist];
  __shared__ int smax, smore;
  if (pass > 0 &&
      __hip_atomic_load(&hdr[kHdrJump + pass], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    return;
  for (int i = threadIdx.x; i < kJumpHist; i += blockDim.x) hist[i] = 0;
  if (threadIdx.x == 0) smax = smore = 0;
  __syncthreads();
  const int n = hdr[1];
  int32_t *counts = hdr + kHdrInts;
  int local_max = 0, more = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = list[i];
    if (__hip_atomic_load(&depth[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0xFFFF)
      continue;
    const unsigned long long j =
        __hip_atomic_load(&jump[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int a = static_cast<int>(j & 0xffffffffu);
    const unsigned d = static_cast<unsigned>(j >> 32);
    const unsigned da = __hip_atomic_load(&depth[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (da != 0xFFFF) {
      const unsigned nd = d + da;
      if (nd > FS_MAX_LEVELS) {
        atomicOr(&hdr[2], kErrDepth);
        continue;
      }
      __hip_atomic_store(&depth[c], static_cast<uint16_t>(nd), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      if (nd < static_cast<unsigned>(kJumpHist)) atomicAdd(&hist[nd], 1);
      else atomicAdd(&counts[nd], 1);
      local_max = max(local_max, static_cast<int>(nd));
    } else {
      const unsigned long long ja =
          __hip_atomic_load(&jump[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned nd = d + static_cast<unsigned>(ja >> 32);
      if (nd > FS_MAX_LEVELS + 1u) {
        atomicOr(&hdr[2], kErrDepth);
        continue;
      }
      __hip_atomic_store(&jump[c],
                         (static_cast<unsigned long long>(nd) << 32) | (ja & 0xffffffffu),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      more = 1;
    }
  }
  if (local_max > 0) atomicMax(&smax, local_max);
  if (more) smore = 1;
  __syncthreads();
  const int top = min(smax, kJumpHist - 1);
  for (int i = threadIdx.x; i <= top; i += blockDim.x)
    if (hist[i]) atomicAdd(&counts[i], hist[i]);
  if (threadIdx.x == 0) {
    if (smax > 0) atomicMax(&hdr[0], smax);
    if (smore)
      __hip_atomic_store(&hdr[kHdrJump + pass + 1], 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Level 0 of GenerateOrder (RB:223-226): every NO_FLOW cell, ring 0
// included, in ascending index.  One tile = 4096 cells, 16 per thread read
// as one 16-byte load.
__global__ __launch_bounds__(kScanBlock) void k_roots(
    const uint8_t *__restrict__ rcv, int32_t *__restrict__ stack, uint64_t *status,
    unsigned long long *ticket, unsigned long long tbase, uint32_t epoch, int32_t N,
    int32_t *hdr) {
  __shared__ uint32_t sh[kScanBlock / kWave + 1];
  __shared__ uint32_t s_tile, s_pre;
  if (threadIdx.x == 0) s_tile = static_cast<uint32_t>(atomicAdd(ticket, 1ull) - tbase);
  __syncthreads();
  const uint32_t tile = s_tile;
  const long long base = static_cast<long long>(tile) * kRootTile +
                         static_cast<long long>(threadIdx.x) * kRootItems;
  uint32_t flags = 0;
  if (base + kRootItems <= N) {
    const uint4 v = *reinterpret_cast<const uint4 *>(rcv + base);
    const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int b = 0; b < 4; b++)
        if (((w4[k] >> (8 * b)) & 0xFFu) == kNoFlow) flags |= 1u << (4 * k + b);
  } else {
    for (int i = 0; i < kRootItems; i++)
      if (base + i < N && rcv[base + i] == kNoFlow) flags |= 1u << i;
  }
  uint32_t total;
  const uint32_t ex = block_excl_scan<kScanBlock>(__popc(flags), &total, sh);
  if (threadIdx.x < kWave) {
    const uint32_t pre = lookback(status, tile, epoch, total, &hdr[2]);
    if (threadIdx.x == 0) s_pre = pre;
  }
  __syncthreads();
  long long pos = static_cast<long long>(s_pre) + ex;
  while (flags) {
    const int i = __builtin_ctz(flags);
    flags &= flags - 1;
    if (pos < N) stack[pos] = static_cast<int32_t>(base + i);
    pos++;
  }
}

// Stack-order records of the level path, written as the breadth-first
// order is built: for stack position p, fdon[p] is where its donor list was
// appended and ndon[p] its length; for every appended donor, rdir is its
// receiver direction 0..7 (RB:79-82).  The donor in mask slot j drains in
// direction kSlotDir[j] (slot 0, the north-west neighbour, drains south-east
// and so on).
__device__ __forceinline__ int slot_dir(int j) {
  constexpr uint32_t kSlotDir = 5u | 6u << 3 | 7u << 6 | 4u << 9 | 0u << 12 | 3u << 15 |
                                2u << 18 | 1u << 21;
  return static_cast<int>((kSlotDir >> (3 * j)) & 7u);
}

__device__ __forceinline__ void append_donors(int32_t c, uint32_t m, int32_t p, long long pos,
                                              int32_t *__restrict__ stack,
                                              uint8_t *__restrict__ rdir,
                                              int32_t *__restrict__ fdon,
                                              uint8_t *__restrict__ ndon, int W, int32_t N) {
  fdon[p] = static_cast<int32_t>(pos < N ? pos : N);
  ndon[p] = static_cast<uint8_t>(__popc(m));
  while (m) {
    const int j = __builtin_ctz(m);
    m &= m - 1;
    if (pos < N) {
      stack[pos] = c + slot_offset(j, W);
      rdir[pos] = static_cast<uint8_t>(slot_dir(j));
    }
    pos++;
  }
}

// One BFS level of GenerateOrder (RB:234-247): stack[ls, le) -> the donor
// lists of those cells, in order, written from stack[le].
__global__ __launch_bounds__(kScanBlock) void k_bfs(
    int32_t *__restrict__ stack, const uint8_t *__restrict__ dmask, uint8_t *__restrict__ rdir,
    int32_t *__restrict__ fdon, uint8_t *__restrict__ ndon, int32_t ls, int32_t le, int W,
    int32_t N, uint64_t *status, unsigned long long *ticket, unsigned long long tbase,
    uint32_t epoch, int32_t *hdr) {
  __shared__ uint32_t sh[kScanBlock / kWave + 1];
  __shared__ uint32_t s_tile, s_pre;
  if (threadIdx.x == 0) s_tile = static_cast<uint32_t>(atomicAdd(ticket, 1ull) - tbase);
  __syncthreads();
  const uint32_t tile = s_tile;
  const long long p0 = static_cast<long long>(ls) + static_cast<long long>(tile) * kBfsTile +
                       static_cast<long long>(threadIdx.x) * kBfsItems;
  int32_t cell[kBfsItems];
  unsigned long long masks = 0;
  uint32_t cnt = 0;
#pragma unroll
  for (int i = 0; i < kBfsItems; i++) {
    const long long p = p0 + i;
    int32_t c = 0;
    uint32_t m = 0;
    if (p < le) {
      c = stack[p];
      if (static_cast<uint32_t>(c) < static_cast<uint32_t>(N)) m = dmask[c];
      else atomicOr(&hdr[2], kErrIndex);
    }
    cell[i] = c;
    masks |= static_cast<unsigned long long>(m) << (8 * i);
    cnt += __popc(m);
  }
  uint32_t total;
  const uint32_t ex = block_excl_scan<kScanBlock>(cnt, &total, sh);
  if (threadIdx.x < kWave) {
    const uint32_t pre = lookback(status, tile, epoch, total, &hdr[2]);
    if (threadIdx.x == 0) s_pre = pre;
  }
  __syncthreads();
  long long pos = static_cast<long long>(le) + s_pre + ex;
#pragma unroll
  for (int i = 0; i < kBfsItems; i++) {
    const long long p = p0 + i;
    if (p >= le) break;
    const uint32_t m = static_cast<uint32_t>(masks >> (8 * i)) & 0xFFu;
    append_donors(cell[i], m, static_cast<int32_t>(p), pos, stack, rdir, fdon, ndon, W, N);
    pos += __popc(m);
  }
}

// Levels [L0, L1) of the BFS in one workgroup, for runs of small levels.
__global__ __launch_bounds__(kSmallBlock) void k_bfs_small(
    int32_t *__restrict__ stack, const uint8_t *__restrict__ dmask, uint8_t *__restrict__ rdir,
    int32_t *__restrict__ fdon, uint8_t *__restrict__ ndon, const int32_t *__restrict__ levels,
    int L0, int L1, int W, int32_t N, int32_t *hdr) {
  __shared__ uint32_t sh[kSmallBlock / kWave + 1];
  for (int L = L0; L < L1; L++) {
    const int32_t ls = levels[L], le = levels[L + 1];
    long long out = le;
    for (long long b = ls; b < le; b += kSmallLevel) {
      const long long p0 = b + static_cast<long long>(threadIdx.x) * kSmallItems;
      int32_t cell[kSmallItems];
      uint32_t masks = 0, cnt = 0;
#pragma unroll
      for (int i = 0; i < kSmallItems; i++) {
        const long long p = p0 + i;
        int32_t c = 0;
        uint32_t m = 0;
        if (p < le) {
          c = stack[p];
          if (static_cast<uint32_t>(c) < static_cast<uint32_t>(N)) m = dmask[c];
          else atomicOr(&hdr[2], kErrIndex);
        }
        cell[i] = c;
        masks |= m << (8 * i);
        cnt += __popc(m);
      }
      uint32_t total;
      const uint32_t ex = block_excl_scan<kSmallBlock>(cnt, &total, sh);
      long long pos = out + ex;
#pragma unroll
      for (int i = 0; i < kSmallItems; i++) {
        const long long p = p0 + i;
        if (p >= le) break;
        const uint32_t m = (masks >> (8 * i)) & 0xFFu;
        append_donors(cell[i], m, static_cast<int32_t>(p), pos, stack, rdir, fdon, ndon, W, N);
        pos += __popc(m);
      }
      out += total;
    }
    __syncthreads();
  }
}

// Upstream cell count of stack entry p: 1 + the counts of its donors, one
// level higher, already final and contiguous from fdon[p].  Counts are kept
// in stack order (cnt_s); accum = count * cell_area exactly (RB:262-279:
// every partial sum there is an integer multiple of cell_area).  Entries of
// the deepest level have no donors (the breadth-first pass never records
// them): top is true for those.
__device__ __forceinline__ void flowacc_entry(int32_t p, bool top,
                                              const int32_t *__restrict__ fdon,
                                              const uint8_t *__restrict__ ndon, uint32_t *cnt_s,
                                              int32_t N, int32_t *hdr) {
  if (top) {
    cnt_s[p] = 1;
    return;
  }
  const int32_t f = fdon[p];
  const int k = ndon[p];
  uint32_t s = 1;
  if (f > p && static_cast<long long>(f) + k <= N) {
    for (int i = 0; i < k; i++) s += cnt_s[f + i];
  } else if (k > 0) {
    atomicOr(&hdr[2], kErrIndex);
  }
  cnt_s[p] = s;
}

__global__ __launch_bounds__(256) void k_flowacc(const int32_t *__restrict__ fdon,
                                                 const uint8_t *__restrict__ ndon,
                                                 uint32_t *cnt_s, int32_t ls, int32_t le,
                                                 bool top, int32_t N, int32_t *hdr) {
  const long long p = static_cast<long long>(ls) + blockIdx.x * 256ll + threadIdx.x;
  if (p >= le) return;
  flowacc_entry(static_cast<int32_t>(p), top, fdon, ndon, cnt_s, N, hdr);
}

// Levels L_hi down to L_lo (inclusive) in one workgroup; L_top is the
// deepest level of the step.
__global__ __launch_bounds__(kSmallBlock) void k_flowacc_small(
    const int32_t *__restrict__ fdon, const uint8_t *__restrict__ ndon, uint32_t *cnt_s,
    const int32_t *__restrict__ levels, int L_hi, int L_lo, int L_top, int32_t N,
    int32_t *hdr) {
  for (int L = L_hi; L >= L_lo; L--) {
    const int32_t ls = levels[L], le = levels[L + 1];
    for (long long p = ls + threadIdx.x; p < le; p += kSmallBlock)
      flowacc_entry(static_cast<int32_t>(p), L == L_top, fdon, ndon, cnt_s, N, hdr);
    __syncthreads();
  }
}

// AddUplift (RB:285-296) for the interior outlets (level-0 cells away from
// rings 0 and 1).  Interior cells with a receiver are uplifted in k_erode.
__global__ __launch_bounds__(256) void k_uplift_roots(const int32_t *__restrict__ stack,
                                                      int32_t n0, double *h, int W, int H,
                                                      double ud, int32_t N, int32_t *hdr) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n0) return;
  const int32_t c = stack[p];
  if (static_cast<uint32_t>(c) >= static_cast<uint32_t>(N)) {
    atomicOr(&hdr[2], kErrIndex);
    return;
  }
  const int y = c / W, x = c - y * W;
  if (x >= 2 && x < W - 2 && y >= 2 && y < H - 2) h[c] += ud;
}

// Plain 16-byte-per-thread copy, used only to calibrate hardware traffic
// counters against a kernel whose HBM bytes are known exactly.
__global__ __launch_bounds__(256) void k_copy_calibration(const uint4 *__restrict__ src,
                                                          uint4 *__restrict__ dst, size_t n) {
  for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += gridDim.x * 256ull)
    dst[i] = src[i];
}

struct ErodeConst {
  double kdt;       // keq*dt
  double lenpow0;   // pow(dx, neq)        cardinal receiver
  double lenpow1;   // pow(dx*SQRT2, neq)  diagonal receiver
  double ud;        // ueq*dt
  double neq;
  double tol;
};

// Per-model constants of the erosion (RB:313-315) and the pow mode of neq.
inline ErodeConst make_erode_const(const fs_params &p, int *nmode) {
  ErodeConst k;
  k.kdt = p.keq * p.dt;
  k.lenpow0 = std::pow(p.dx, p.neq);
  k.lenpow1 = std::pow(p.dx * fs::kSqrt2, p.neq);
  k.ud = p.ueq * p.dt;
  k.neq = p.neq;
  k.tol = p.tol;
  // the short forms of the solve take at least one iteration; with an infinite
  // tolerance the reference's loop takes none, and neither does mode 0's
  *nmode = !std::isfinite(p.tol) ? 0 : (p.neq == 1.0) ? 1 : (p.neq == 2.0) ? 2 : 0;
  return k;
}

// v_min_f64 and v_max_f64 as they are, without the instruction per operand that
// fmin and fmax spend on quieting signalling NaNs
__device__ __forceinline__ double raw_min(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double raw_max(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// The implicit update of one cell (RB:313-326), operation for operation.
// NMODE 1: n = 1, where libm returns pow(x,1) = x and pow(x,0) = 1 exactly;
// NMODE 2: n = 2 with x*x for pow(x,2); NMODE 0: any n through the device
// pow.  fact = (K*dt)*A^m / dr^n, h0 is the uplifted elevation h + U*dt
// (RB:294) and hn the receiver's final elevation.
template <int NMODE>
__device__ __forceinline__ double newton_plain(double h0, double hn, double fact,
                                               const ErodeConst &k, int32_t *hdr) {
  double hnew = h0, hp = h0, diff = 2.0 * k.tol;
  int it = 0;
  while (fabs(diff) > k.tol) {
    const double x = hnew - hn;
    double p1, p0;
    if (NMODE == 1) {
      p1 = x;
      p0 = 1.0;
    } else if (NMODE == 2) {
      p1 = x * x;
      p0 = x;
    } else {
      p1 = pow(x, k.neq);
      p0 = pow(x, k.neq - 1.0);
    }
    hnew = hnew - ((hnew - h0) + fact * p1) / (1.0 + (fact * k.neq) * p0);
    diff = hnew - hp;
    hp = hnew;
    if (++it >= kNewtonCap) {
      atomicOr(&hdr[2], kErrNewton);
      break;
    }
  }
  return hnew;
}

// The same update with the same bits in fewer instructions: solves wait for
// each other along drainage paths (245 cells and 2171 Newton iterations on the
// deepest one at 501^2 with the reference's constants), and a wave that runs
// alone is bound by its instruction count, scalar ones included.  A solve by
// one wave takes 92 ns against 248 for n = 1, 76 ns against 94 per iteration for
// n = 2.
//
// Division.  For operands far from the ends of the exponent range, an IEEE
// division a / b is, on this hardware, the refined reciprocal y of b
// (v_rcp_f64 and two Newton-Raphson steps), q = a*y, and the correction q +
// (a - b*q)*y; what else the compiler emits for it scales operands near the
// ends of the range and does nothing here.  So the quotient is the one the
// plain loop gets, and y does not depend on a: for n = 1 it is ready before
// the receiver is.
//
// Range.  n = 1: with |h0|, |hn| <= 2^200 and 0 <= fact <= 2^200 no operand is
// too large.  n = 2: with |hn| <= h0 <= 2^20 and 0 <= fact*n <= 2^28, the
// iterates fall from h0 towards the root, which is not below hn; rounding can
// take one below hn by 2^-29 at most (8 ulps of h0 - hn), so every denominator
// is at least 1/2.  A numerator may still be too small (or zero): then its
// quotient is below 2^-400, the iteration ends the solve, and h - q is h
// whatever the quotient's last bits, unless h is tiny too.  So a result of at
// least 2^-290 is the plain loop's; every other cell (NaN and infinities among
// them) goes through the plain loop.
//
// Control.  n = 1 is linear: the second iteration confirms the first.  n = 2
// takes kNewtonFirst iterations before the wave first looks whether all its
// lanes have converged (nearly every cell needs five to seven); a lane keeps
// the iterate at which its own loop would have ended.  The iteration at which
// the plain loop fails, converged or not, is left to it.
__device__ __forceinline__ double refined_rcp(double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
}
__device__ __forceinline__ double quotient(double a, double b, double y) {
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}
constexpr double kNewtonLarge = 0x1p200, kNewtonSmall = 0x1p-290;
constexpr int kNewtonFirst = 6;

// What a solve can do before its receiver is known.
struct NewtonPrep {
  double b, y;   // n = 1: the denominator and its reciprocal
  double fn;     // fact * n
  double zero;   // h0 - h0
  bool ok;       // h0 and fact are in range
};
template <int NMODE>
__device__ __forceinline__ NewtonPrep newton_prep(double h0, double fact, const ErodeConst &k) {
  NewtonPrep p;
  p.fn = fact * k.neq;
  p.zero = h0 - h0;
  p.b = 1.0 + p.fn;
  p.y = NMODE == 1 ? refined_rcp(p.b) : 0.0;
  if constexpr (NMODE == 2) p.ok = h0 <= 0x1p20 && fact >= 0.0 && p.fn <= 0x1p28;
  else p.ok = fabs(h0) <= kNewtonLarge && fact >= 0.0 && fact <= kNewtonLarge;
  return p;
}

template <int NMODE>
__device__ __forceinline__ double newton_solve(double h0, double hn, double fact,
                                               const NewtonPrep &p, const ErodeConst &k,
                                               int32_t *hdr) {
  if constexpr (NMODE == 1) {
    const double a1 = p.zero + fact * (h0 - hn);
    const double h1 = h0 - quotient(a1, p.b, p.y);
    const double d1 = h1 - h0;
    const double a2 = d1 + fact * (h1 - hn);
    const double h2 = h1 - quotient(a2, p.b, p.y);
    const bool one = !(fabs(d1) > k.tol), two = !(fabs(h2 - h1) > k.tol);
    const double res = one ? h1 : h2;
    if (p.ok & (fabs(hn) <= kNewtonLarge) & (fabs(res) >= kNewtonSmall) & (one | two)) return res;
    return newton_plain<1>(h0, hn, fact, k, hdr);
  } else if constexpr (NMODE == 2) {
    double h = h0, res = h0;
    bool done = false;
    auto iterate = [&]() {
      const double x = h - hn;
      const double b = 1.0 + p.fn * x;
      const double a = (h - h0) + fact * (x * x);
      const double hnew = h - quotient(a, b, refined_rcp(b));
      res = done ? res : hnew;
      done = done | !(fabs(hnew - h) > k.tol);
      h = hnew;
    };
#pragma unroll
    for (int it = 0; it < kNewtonFirst; it++) iterate();
#pragma nounroll
    for (int it = kNewtonFirst; it < kNewtonCap - 1 && __ballot(!done) != 0; it++) iterate();
    if (p.ok & done & (fabs(hn) <= h0) & (fabs(res) >= kNewtonSmall)) return res;
    return newton_plain<2>(h0, hn, fact, k, hdr);
  } else {
    return newton_plain<NMODE>(h0, hn, fact, k, hdr);
  }
}

template <int NMODE>
__device__ __forceinline__ double newton_update(double h0, double hn, double fact,
                                                const ErodeConst &k, int32_t *hdr) {
  if constexpr (NMODE == 1)
    return newton_solve<1>(h0, hn, fact, newton_prep<1>(h0, fact, k), k, hdr);
  return newton_plain<NMODE>(h0, hn, fact, k, hdr);
}

// Erode for stack entry p (RB:306-328): the cell's new elevation from
// h + U*dt and its receiver's final elevation (one level lower, so already
// written; it sits next to the cell in the grid, usually in the same cache
// line).  The count and the receiver direction come from stack order.
template <int NMODE>
__device__ __forceinline__ void erode_entry(int32_t p, const int32_t *__restrict__ stack,
                                            const uint8_t *__restrict__ rdir,
                                            const uint32_t *__restrict__ cnt_s,
                                            const double *__restrict__ ftab, double *h, int W,
                                            int32_t N, const ErodeConst &k, int32_t *hdr) {
  const int32_t c = stack[p];
  const int r = rdir[p] & 7;
  uint32_t a = cnt_s[p];
  const int32_t nb = c + dir_offset(r, W);
  if (static_cast<uint32_t>(c) >= static_cast<uint32_t>(N) ||
      static_cast<uint32_t>(nb) >= static_cast<uint32_t>(N) || a > static_cast<uint32_t>(N)) {
    atomicOr(&hdr[2], kErrIndex);
    return;
  }
  h[c] = newton_update<NMODE>(h[c] + k.ud, h[nb], ftab[2 * a + (r & 1)], k, hdr);
}

template <int NMODE>
__global__ __launch_bounds__(256) void k_erode(const int32_t *__restrict__ stack,
                                               const uint8_t *__restrict__ rdir,
                                               const uint32_t *__restrict__ cnt_s,
                                               const double *__restrict__ ftab, double *h,
                                               int32_t ls, int32_t le, int W, int32_t N,
                                               ErodeConst k, int32_t *hdr) {
  const long long p = static_cast<long long>(ls) + blockIdx.x * 256ll + threadIdx.x;
  if (p >= le) return;
  erode_entry<NMODE>(static_cast<int32_t>(p), stack, rdir, cnt_s, ftab, h, W, N, k, hdr);
}

template <int NMODE>
__global__ __launch_bounds__(kSmallBlock) void k_erode_small(
    const int32_t *__restrict__ stack, const uint8_t *__restrict__ rdir,
    const uint32_t *__restrict__ cnt_s, const double *__restrict__ ftab, double *h,
    const int32_t *__restrict__ levels, int L_lo, int L_hi, int W, int32_t N, ErodeConst k,
    int32_t *hdr) {
  for (int L = L_lo; L <= L_hi; L++) {
    const int32_t ls = levels[L], le = levels[L + 1];
    for (long long p = ls + threadIdx.x; p < le; p += kSmallBlock)
      erode_entry<NMODE>(static_cast<int32_t>(p), stack, rdir, cnt_s, ftab, h, W, N, k, hdr);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// depression filling (an extension: the reference has none)
// ---------------------------------------------------------------------------
// The Priority-Flood+epsilon surface (Barnes, Lehman & Mulla 2014): the
// unique fixed point of F = max(h, nextafter(min over the D8 neighbours of F,
// +inf)) on interior cells, rings 0 and 1 held at h.  Starting from +inf the
// update only lowers F, so tiles relax it in LDS against their neighbours'
// last values (reads may see older, higher values: the iteration still
// decreases to the fixed point); the host relaunches until a launch changes
// nothing, which leaves every cell consistent with its neighbours' final
// values.
constexpr int kFillTile = 64;
constexpr int kFillReg = kFillTile + 2;
constexpr int kFillBlock = 1024;
constexpr int kFillInner = 6;             // a wave's relaxations between two votes of the block
constexpr int kFillVotes = 4096;          // votes per launch at most

// nextafter(x, +inf) for IEEE doubles.
__device__ __forceinline__ double next_up(double x) {
  if (!(x < __builtin_huge_val())) return x;          // +inf, NaN
  if (x == 0.0) return 0x1p-1074;                      // +-0 -> smallest subnormal
  const long long u = __double_as_longlong(x);
  return __longlong_as_double(x > 0.0 ? u + 1 : u - 1);
}

// F = h on rings 0 and 1, +inf inside.
__global__ __launch_bounds__(256) void k_fill_init(const double *__restrict__ h,
                                                   double *__restrict__ F, int W, int H) {
  const long long N = static_cast<long long>(W) * H;
  for (long long c = blockIdx.x * 256ll + threadIdx.x; c < N; c += gridDim.x * 256ll) {
    const int y = static_cast<int>(c / W), x = static_cast<int>(c - static_cast<long long>(y) * W);
    const bool inner = x >= 2 && x < W - 2 && y >= 2 && y < H - 2;
    F[c] = inner ? __builtin_huge_val() : h[c];
  }
}

// One tile: relaxed to its fixed point in LDS, its border published and the
// neighbours' borders read again, until such a read brings nothing new.
//
// A flood path runs cell by cell and values are corrected several times on
// the way, so the time is a chain of relaxations.  Each wave owns a patch of 16
// x 16 cells and relaxes 2 x 2 of them per lane from LDS, up to kFillInner
// times between two votes of the workgroup, with no barrier in between: values
// only fall, and any order ends at the same fixed point.  A wave whose patch
// and whose neighbours have no news rests, which leaves LDS to the others.
// 256 threads with 16 strided cells each and three barriers a sweep took 266
// us per launch on a random 700 x 501 terrain and 7.9 ms for the fill; this
// takes 2.5 (5.0 ms against 16.5 at 1000^2, 14.0 against 37.4 at 3000 x 2000).
// Two relaxations between votes: 3.2 ms, 16: 2.7; waiting in the launch for
// further news (40 more reads): 3.0.
__global__ __launch_bounds__(kFillBlock) void k_fill(const double *__restrict__ h, double *F,
                                                     int W, int H, int tiles_x,
                                                     const int32_t *before, int32_t *changed) {
  // the launch before found every tile settled
  if (before != nullptr && *before == 0) return;
  __shared__ double f_s[kFillReg * kFillReg];
  __shared__ uint32_t dirty;   // patches with news, one bit per wave
  const int x0 = (blockIdx.x % tiles_x) * kFillTile, y0 = (blockIdx.x / tiles_x) * kFillTile;
  if (threadIdx.x == 0) dirty = 0xFFFFu;
  auto load_f = [&](int gx, int gy) {
    return (gx >= 0 && gx < W && gy >= 0 && gy < H)
               ? __builtin_canonicalize(__hip_atomic_load(&F[static_cast<size_t>(gy) * W + gx],
                                                          __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT))
               : __builtin_huge_val();
  };
  for (int i = threadIdx.x; i < kFillReg * kFillReg; i += kFillBlock)
    f_s[i] = load_f(x0 - 1 + i % kFillReg, y0 - 1 + i / kFillReg);
  // this lane's 2 x 2 cells
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int lx = (wave % 4) * 16 + (lane % 8) * 2, ly = (wave / 4) * 16 + (lane / 8) * 2;
  double hv[2][2];
  bool inner[2][2];
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int gx = x0 + lx + i, gy = y0 + ly + j;
      inner[j][i] = gx >= 2 && gx < W - 2 && gy >= 2 && gy < H - 2;
      hv[j][i] = inner[j][i] ? __builtin_canonicalize(h[static_cast<size_t>(gy) * W + gx]) : 0.0;
    }
  // the halo cell this thread looks after: the ring around the tile
  constexpr int kRing = 4 * kFillReg - 4;
  static_assert(kRing <= kFillBlock, "one halo cell per thread");
  int halo = -1, hx = 0, hy = 0;
  if (static_cast<int>(threadIdx.x) < kRing) {
    const int q = threadIdx.x;
    if (q < kFillReg) {
      hx = q;
    } else if (q < 2 * kFillReg) {
      hx = q - kFillReg;
      hy = kFillReg - 1;
    } else {
      hx = q < 3 * kFillReg - 2 ? 0 : kFillReg - 1;
      hy = (q - 2 * kFillReg) % (kFillReg - 2) + 1;
    }
    halo = hy * kFillReg + hx;
  }
  const bool border = lx == 0 || ly == 0 || lx + 2 == kFillTile || ly + 2 == kFillTile;
  auto ld = [&](int i) {
    return __hip_atomic_load(&f_s[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto st = [&](int i, double v) {
    __hip_atomic_store(&f_s[i], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  // news is published behind the values it stands for, and taken before they are
  // read
  auto publish = [&](uint32_t patches) {
    __hip_atomic_fetch_or(&dirty, patches, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto take = [&](uint32_t patch) {
    return __hip_atomic_fetch_and(&dirty, ~patch, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) &
           patch;
  };
  const int c0 = (ly + 1) * kFillReg + lx + 1;
  // the patches around this wave's
  uint32_t around = 0;
#pragma unroll
  for (int j = -1; j < 2; j++)
#pragma unroll
    for (int i = -1; i < 2; i++) {
      const int px = wave % 4 + i, py = wave / 4 + j;
      if ((i || j) && px >= 0 && px < 4 && py >= 0 && py < 4) around |= 1u << (4 * py + px);
    }
  // the lane's cells, which it alone writes
  double own[2][2];
  // one relaxation of them; true when one fell
  auto relax = [&]() {
    double f[4][4];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        f[j][i] = j % 3 && i % 3 ? own[(j - 1) & 1][(i - 1) & 1]
                                 : ld(c0 + (j - 1) * kFillReg + i - 1);
    bool fell = false;
#pragma unroll
    for (int j = 1; j < 3; j++)
#pragma unroll
      for (int i = 1; i < 3; i++) {
        const double a = raw_min(raw_min(f[j - 1][i - 1], f[j - 1][i]), f[j - 1][i + 1]);
        const double b = raw_min(raw_min(f[j + 1][i - 1], f[j + 1][i]), f[j + 1][i + 1]);
        const double m = raw_min(raw_min(a, b), raw_min(f[j][i - 1], f[j][i + 1]));
        const double v = raw_max(hv[j - 1][i - 1], next_up(m));
        if (inner[j - 1][i - 1] && v < f[j][i]) {
          f[j][i] = own[j - 1][i - 1] = v;
          fell = true;
          st(c0 + (j - 1) * kFillReg + i - 1, v);
        }
      }
    return fell;
  };
  auto store_cells = [&]() {
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int i = 0; i < 2; i++)
        if (inner[j][i])
          __hip_atomic_store(&F[static_cast<size_t>(y0 + ly + j) * W + x0 + lx + i],
                             own[j][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  // the neighbours' cell this thread looks after, read again; its news wakes
  // the patches it touches
  auto halo_news = [&]() {
    if (halo < 0) return 0;
    const double v = load_f(x0 - 1 + hx, y0 - 1 + hy);
    if (!(v < ld(halo))) return 0;
    st(halo, v);
    uint32_t wake = 0;
    for (int j = -1; j < 2; j++)
      for (int i = -1; i < 2; i++) {
        const int cx = hx - 1 + i, cy = hy - 1 + j;
        if (cx >= 0 && cx < kFillTile && cy >= 0 && cy < kFillTile)
          wake |= 1u << (4 * (cy / 16) + cx / 16);
      }
    publish(wake);
    return 1;
  };
  bool ever = false;        // block-uniform: a cell fell in this launch
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 2; i++) own[j][i] = ld(c0 + j * kFillReg + i);
  for (int votes = 0; votes < kFillVotes;) {
    bool moved = false;     // block-uniform: since the last publication
    for (; votes < kFillVotes; votes++) {
      // a wave rests while neither it nor a patch around it has news
      int fell = 0;
      uint32_t mine = 0;
      if (lane == 0) mine = take(1u << wave);
      if (__builtin_amdgcn_readfirstlane(mine)) {
        bool now = true;
        for (int k = 0; k < kFillInner && __any(now); k++) {
          now = relax();
          fell |= now ? 1 : 0;
        }
        const uint32_t wake = (__any(fell) ? around : 0u) | (__any(now) ? 1u << wave : 0u);
        if (wake != 0 && lane == 0) publish(wake);
      }
      if (!__syncthreads_or(fell)) break;
      moved = true;
    }
    if (moved) {
      ever = true;
      if (border) store_cells();
    }
    votes++;
    if (!__syncthreads_or(halo_news())) break;
  }
  if (!ever) return;
  store_cells();
  if (threadIdx.x == 0) atomicOr(changed, 1);
}

// ---------------------------------------------------------------------------
// phase timing of the tile kernels
// ---------------------------------------------------------------------------
// The tile path fuses the reference's stages (donors, order, accumulation,
// uplift, erosion; RB:367-372) into two kernels.  To report the reference's
// per-stage timers, the timed instantiations of the tile kernels (run on a
// sample of steps) let one workgroup in kPhaseSample add the wall-clock
// ticks of each of its phases (between barriers, never inside a loop:
// reading the clock is a slow scalar-memory access) to a row of `phase`
// (rows spread the atomics); the host splits the kernels' event times over
// the stages in proportion.
constexpr int kPhaseSample = 16;     // workgroups per sampled one in a timed launch
constexpr int kPhaseEvery = 32;      // tile steps per timed step
constexpr int kPhaseSlots = 32;
constexpr int kPhaseStride = 8;
constexpr size_t kPhaseWords = static_cast<size_t>(kPhaseSlots) * kPhaseStride;
enum PhaseId {
  kPhAccLoad = 0,    // receivers -> region words (the donor structure)   Donors
  kPhAccWalk,        // receiver-chain walks: counts and levels          FlowAcc
  kPhAccPlan,        // halo chains, slot scan, erosion plan             Order
  kPhAccStore,       // count and level stores                           FlowAcc
  kPhEroBucket,      // loads and level bucketing of the slots           Order
  kPhEroRoots,       // uplift of the outlets                            Uplift
  kPhEroLoop,        // the erosion wavefront                            Erosion
  kPhEroStore,       // elevation stores                                 Erosion
  kPhCount
};
static_assert(kPhCount <= kPhaseStride, "phase row");

// This workgroup's phase row, or null when it is not sampled.  Workgroups go to
// the eight XCDs in turn: eight in a row are sampled, one on each.
__device__ __forceinline__ unsigned long long *phase_row(unsigned long long *phase) {
  const unsigned turn = blockIdx.x / 8;
  if (!phase || turn % kPhaseSample != 0) return nullptr;
  return phase + (8 * (turn / kPhaseSample) + blockIdx.x % 8) % kPhaseSlots * kPhaseStride;
}
// A sampled workgroup's clock at its k-th phase boundary, kept in LDS: in scalar
// registers the times took the timed erosion from 70 to 82 of them, and beyond 80
// a CU holds one workgroup of 1024 threads instead of two (1039 us against 610
// at 10000 x 10000; with the times in LDS 609).
__device__ __forceinline__ void phase_mark(const unsigned long long *row, uint64_t *clock, int k) {
  if (row && threadIdx.x == 0) clock[k] = wall_clock64();
}
// Ends the last of the phases first .. first + 3, and adds them to the row.
__device__ __forceinline__ void phase_end(unsigned long long *row, uint64_t *clock, int first) {
  if (row && threadIdx.x == 0) {
    clock[4] = wall_clock64();
    for (int k = 0; k < 4; k++) atomicAdd(&row[first + k], clock[k + 1] - clock[k]);
  }
}

// ---------------------------------------------------------------------------
// tile path, 16-cell halo (fs_tile.h)
// ---------------------------------------------------------------------------
#define FS_TILE_HALO 16
#include "fs_tile.h"
#undef FS_TILE_HALO

}  // namespace

#endif
