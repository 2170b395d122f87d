// fs_ensemble.hip -- many FastScape grids ("realizations") of different
// sizes and parameters advanced together, every kernel of a time-step
// launched once for all of them.
//
// Every realization takes the reference's time-step (fastscape_RB.cpp:366-376)
// and gets the same bits as a single-grid model with its size, parameters and
// initial terrain.  A step, on one stream:
//
//   k_ens_receivers  receivers of every realization (RB:160-182)
//   k_ens_acc        tile accumulation (upstream counts and levels,
//                    RB:213-279) of every 64x64 tile of the candidates: the
//                    realizations at most kHalo levels deep last step; a tile
//                    deeper than kHalo marks its realization deep
//   k_ens_lists      one workgroup: each realization's path this step, and the
//                    deep ones' tiles as the tile-graph kernels' work list
//   k_ens_erode      tile uplift + erosion (RB:285-328) of the others
//
// The deep realizations then take one tile-graph step together (fs_deep.h):
// per 64x64 tile with no halo, every deep realization's tiles in the same
// launches, the tiles joined by the graph of the cells where drainage leaves
// a tile; the step also counts their levels, so the next step knows which
// are shallow again.  The host reads the work list's size while k_ens_erode
// runs.
//
// The kernels are the single-grid ones' bodies, with a table from workgroup to
// realization; workgroups of realizations on the other path return at once.
// One persistent cooperative kernel for all phases ran one 1024-thread
// workgroup per CU (the LDS of its largest phase) behind grid barriers: 394 us
// a step for 32 realizations of 256^2 (512 tiles), which these four kernels
// step in 64.
//
// A cell's elevation depends only on its own inputs and its receiver's final
// value, and upstream counts are integers, so the order of the work is free: the
// schedule (fs_schedule) says how much of it a workgroup takes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <new>
#include <numeric>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "fs_internal.h"
#include "fs_hostutil.h"

#include "fs_device.h"
#include "fs_deep.h"

namespace {

constexpr int kEnsBlock = 1024;                     // k_ens_lists
constexpr int kHistLen = kHalo + 1;
constexpr int kRecvRows = 16;                       // schedules name multiples of this
constexpr int kRecvPerBlock = 64;                   // rows named per receiver block
constexpr int kMaxRealizations = 1 << 20;

// per-realization state words (kRH ints each)
constexpr int kRH = 16;
constexpr int kRhDepth = 0;       // deepest level of the last step
constexpr int kRhOver = 1;        // tiles deeper than kHalo this step
constexpr int kRhErr = 2;         // error bits (same slot as a model's hdr[2])
constexpr int kRhPath = 7;        // path of the last step: 1 tiles, 3 tile graph
constexpr int kRhTileSteps = 9;
constexpr int kRhLevelSteps = 10;   // steps off the tiles (the tile graph)

struct EnsReal {
  uint64_t off;        // first cell of the realization in the cell arrays
  uint64_t ftab_off;   // first entry of its erosion factor table
  uint64_t lev_off;    // first entry of its level counts
  uint64_t plan_off;   // first tile plan of the realization
  int W, H, tiles_x, ntiles;
  int lev_cap;         // level entries available
  int nmode;
  int recv_xb;         // receiver column blocks
  int recv_first;      // first receiver workgroup
  double d_card, d_diag;
  ErodeConst ek;
};

// The realizations and their state.
struct EnsArgs {
  const EnsReal *real;
  int R;
  double *h_old, *h_new;
  uint8_t *rcv, *lvl;
  uint32_t *cnt;
  TilePlan *plan;
  const double *ftab;
  int32_t *rh, *hist;
};

// Lists the realizations r in [0, R) with pick(r): real[e] is entry e's
// realization, off[e] its first tile in the list.  One workgroup of kEnsBlock
// threads; sh holds kEnsBlock / kWave + 1 words.
template <class Pick>
__device__ void list_entries(int R, const EnsReal *rl, Pick pick, int32_t *off, int32_t *real,
                             int &entries, int &tiles, uint32_t *sh) {
  entries = tiles = 0;
  for (int base = 0; base < R; base += kEnsBlock) {
    const int r = base + threadIdx.x;
    const int v = r < R && pick(r) ? rl[r].ntiles : 0;
    uint32_t te, ti;
    const uint32_t ee = block_excl_scan<kEnsBlock>(v > 0 ? 1u : 0u, &te, sh);
    const uint32_t ei = block_excl_scan<kEnsBlock>(static_cast<uint32_t>(v), &ti, sh);
    if (v > 0) {
      off[entries + ee] = tiles + static_cast<int>(ei);
      real[entries + ee] = r;
    }
    entries += static_cast<int>(te);
    tiles += static_cast<int>(ti);
  }
}

template <int NM, class F>
__device__ __forceinline__ void with_nmode(int nm, F f) {
  if constexpr (NM >= 0) {
    f(std::integral_constant<int, NM>{});
  } else {
    if (nm == 1) f(std::integral_constant<int, 1>{});
    else if (nm == 2) f(std::integral_constant<int, 2>{});
    else f(std::integral_constant<int, 0>{});
  }
}

// Workgroup number in a grid of ens_grid's shape.
__device__ __forceinline__ int ens_block() {
  return static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x);
}

// Receivers of block b: 64 columns x kRecvShort * kRecvGroups rows of
// realization recv_real[b].
__device__ __forceinline__ void ens_recv_block(const EnsArgs &a,
                                               const int32_t *__restrict__ recv_real, int b) {
  const int r = recv_real[b];
  const EnsReal &g = a.real[r];
  const int local = b - g.recv_first;
  if (local == 0) {   // the realization's per-step state
    if (threadIdx.x == 0) a.rh[static_cast<size_t>(r) * kRH + kRhOver] = 0;
    if (threadIdx.x < kHistLen) a.hist[static_cast<size_t>(r) * kHistLen + threadIdx.x] = 0;
  }
  const int x = (local % g.recv_xb) * kWave + static_cast<int>(threadIdx.x % kWave) + 2;
  const int group = __builtin_amdgcn_readfirstlane((local / g.recv_xb) * kRecvGroups +
                                                   threadIdx.x / kWave);
  if (x >= g.W - 2 || group * kRecvShort + 2 >= g.H - 2) return;
  ShortRows v;
  load_short(v, a.h_old + g.off, g.W, g.H, x, group);
  decide_short(v, a.rcv + g.off, g.W, g.H, x, group, g.d_card, g.d_diag);
}

// A workgroup takes per_group of the nblocks blocks (kMany), or one: the loop
// over them costs registers (92 instead of 76).
template <bool kMany>
__global__ __launch_bounds__(256) void k_ens_receivers(EnsArgs a,
                                                       const int32_t *__restrict__ recv_real,
                                                       int nblocks, int per_group) {
  if constexpr (kMany) {
    const long long first = static_cast<long long>(ens_block()) * per_group;
    const int end = static_cast<int>(min(static_cast<long long>(nblocks), first + per_group));
    for (int b = static_cast<int>(min(first, static_cast<long long>(end))); b < end; b++)
      ens_recv_block(a, recv_real, b);
  } else {
    const int b = ens_block();
    if (b < nblocks) ens_recv_block(a, recv_real, b);
  }
}

// tile_real: each tile's realization (tiles numbered across realizations).
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_ens_acc(EnsArgs a, const int32_t *__restrict__ tile_real,
                                                   int ntiles) {
  __shared__ AccShared sh;
  const int b = ens_block();
  if (b >= ntiles) return;
  const int tile = xcd_tile(b, ntiles);
  const int r = tile_real[tile];
  int32_t *const q = a.rh + static_cast<size_t>(r) * kRH;
  if (q[kRhDepth] > kHalo) return;   // no candidate: it takes the tile graph
  const EnsReal &g = a.real[r];
  const int over = tile_acc_body<BLOCK>(
      sh, a.rcv + g.off, a.cnt + g.off, a.lvl + g.off, a.plan + tile, g.W, g.H,
      tile - static_cast<int>(g.plan_off), g.tiles_x,
      a.hist + static_cast<size_t>(r) * kHistLen, nullptr);
  if (threadIdx.x == 0 && over) atomicAdd(&q[kRhOver], 1);
}

// The path of every realization this step; size[0..1] (and host_size, read by
// the host once this launch has finished): the tile-graph work list's entries
// and tiles.
__global__ __launch_bounds__(kEnsBlock) void k_ens_lists(EnsArgs a, int32_t *tab_off,
                                                         int32_t *tab_real, int32_t *size,
                                                         int32_t *host_size) {
  __shared__ uint32_t sh[kEnsBlock / kWave + 1];
  for (int r = threadIdx.x; r < a.R; r += kEnsBlock) {
    int32_t *const q = a.rh + static_cast<size_t>(r) * kRH;
    int n[kHistLen], D = 0;
#pragma unroll
    for (int l = 0; l < kHistLen; l++) n[l] = a.hist[static_cast<size_t>(r) * kHistLen + l];
#pragma unroll
    for (int l = 0; l < kHistLen; l++) D = n[l] ? l : D;
    if (q[kRhDepth] > kHalo || q[kRhOver] > 0) {
      q[kRhPath] = 3;
      q[kRhLevelSteps]++;
    } else {
      q[kRhDepth] = D;
      q[kRhPath] = 1;
      q[kRhTileSteps]++;
    }
  }
  __syncthreads();
  int entries, tiles;
  list_entries(a.R, a.real, [&](int r) { return a.rh[static_cast<size_t>(r) * kRH + kRhPath] == 3; },
               tab_off, tab_real, entries, tiles, sh);
  if (threadIdx.x == 0) {
    tab_off[entries] = tiles;
    size[0] = entries;
    size[1] = tiles;
    __hip_atomic_store(&host_size[0], entries, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&host_size[1], tiles, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

template <int NM>
__device__ __forceinline__ void ens_erode_tile(EroShared &sh, const EnsArgs &a, int r,
                                               int32_t *q, int tile) {
  const EnsReal &g = a.real[r];
  const ErodeConst ek = g.ek;
  with_nmode<NM>(g.nmode, [&](auto c) {
    tile_erode_body<decltype(c)::value>(sh, a.h_old + g.off, a.h_new + g.off, a.plan + tile,
                                        a.lvl + g.off, a.cnt + g.off, a.ftab + g.ftab_off, g.W,
                                        g.H, tile - static_cast<int>(g.plan_off), g.tiles_x, ek, q);
  });
}

// A workgroup takes per_group of the ntiles tiles, one after another (kMany), or
// one: the loop over them would take 94 registers where two workgroups per CU
// have 64 (held to these it spills 60 bytes a lane).
template <int NM, bool kMany>
__global__ __launch_bounds__(kEroBlock, kMany ? 8 : 1) void k_ens_erode(
    EnsArgs a, const int32_t *__restrict__ tile_real, int ntiles, int per_group) {
  __shared__ EroShared sh;
  const int b = ens_block();
  if constexpr (kMany) {
    const int groups = (ntiles - 1) / per_group + 1;
    if (b >= groups) return;
    const int first = xcd_tile(b, groups) * per_group, n = min(ntiles - first, per_group);
    for (int j = 0; j < n; j++) {
      const int r = tile_real[first + j];
      int32_t *const q = a.rh + static_cast<size_t>(r) * kRH;
      if (q[kRhPath] != 1) continue;
      __syncthreads();   // the LDS of the tile before is free
      ens_erode_tile<NM>(sh, a, r, q, first + j);
    }
  } else {
    if (b >= ntiles) return;
    const int tile = xcd_tile(b, ntiles);
    const int r = tile_real[tile];
    int32_t *const q = a.rh + static_cast<size_t>(r) * kRH;
    if (q[kRhPath] != 1) return;
    ens_erode_tile<NM>(sh, a, r, q, tile);
  }
}

}  // namespace

// ===========================================================================
// host side
// ===========================================================================
struct fs_ensemble {
  int device = 0;
  int R = 0;
  size_t cells = 0;
  hipStream_t stream = nullptr;
  std::vector<fs_realization> spec;   // internal order
  std::vector<int> to_internal;       // user index -> internal index
  std::vector<EnsReal> real;
  int nm_all = -1;                    // shared pow mode, -1 when mixed
  int ncu = 0;

  EnsReal *real_d = nullptr;
  double *h[2] = {nullptr, nullptr};
  uint8_t *rcv = nullptr, *lvl = nullptr;
  uint32_t *cnt = nullptr;
  TilePlan *plan = nullptr;
  int32_t *lev = nullptr;                     // per-level counts of tile-graph steps
  double *ftab = nullptr;
  int32_t *rh = nullptr, *hist = nullptr;
  int32_t *recv_real = nullptr, *tile_real = nullptr;   // workgroup -> realization
  int recv_blocks = 0;
  int tiles = 0;                              // tiles of every realization
  int32_t *tabG_off = nullptr, *tabG_real = nullptr, *tabG_size = nullptr;
  int32_t *graph_n_h = nullptr;               // pinned: the tile-graph work list's size
  hipEvent_t listed = nullptr;                // the list of this step is there
  // the tile-graph step of the deep realizations (fs_deep.h)
  deep::GraphGrid *graph_grid = nullptr;
  uint32_t *dinfo = nullptr, *link = nullptr;
  uint64_t *node_word = nullptr, *items = nullptr;
  uint32_t *node_kids = nullptr, *node_parent = nullptr, *node_out = nullptr;
  uint32_t *node_up = nullptr, *node_level = nullptr;
  int32_t *node_cell = nullptr, *nexit = nullptr, *tile_n0 = nullptr;
  uint16_t *node_tier = nullptr;
  uint32_t *cells_list = nullptr;
  int32_t *thist = nullptr, *tcur = nullptr, *tstat = nullptr;
  int graph_blocks = 0, graph_queues = 1;
  uint64_t graph_tiles = 0;                   // tile-graph tiles stepped so far
  int cur = 0;
  fs_schedule sched{64, 1, 0};
  bool broken = false, have_step = false;
  uint64_t steps = 0;
  double step_ms = 0;
  hipEvent_t ev[2] = {nullptr, nullptr};
  // autotuning
  int tune_trial = 0, tune_interval = 0;
  uint64_t tuned_at = ~0ull;
  std::vector<fs_schedule> tune_cand;
  std::vector<double> tune_ms;
};

namespace {

void free_ensemble(fs_ensemble *e) {
  if (!e) return;
  (void)hipSetDevice(e->device);
  if (e->stream) (void)hipStreamSynchronize(e->stream);
  for (void *p : {static_cast<void *>(e->real_d), static_cast<void *>(e->h[0]),
                  static_cast<void *>(e->h[1]), static_cast<void *>(e->rcv),
                  static_cast<void *>(e->lvl), static_cast<void *>(e->cnt),
                  static_cast<void *>(e->plan), static_cast<void *>(e->lev),
                  static_cast<void *>(e->ftab), static_cast<void *>(e->rh),
                  static_cast<void *>(e->hist), static_cast<void *>(e->recv_real),
                  static_cast<void *>(e->tile_real), static_cast<void *>(e->tabG_off),
                  static_cast<void *>(e->tabG_real), static_cast<void *>(e->tabG_size),
                  static_cast<void *>(e->graph_grid), static_cast<void *>(e->dinfo),
                  static_cast<void *>(e->link), static_cast<void *>(e->node_word),
                  static_cast<void *>(e->items), static_cast<void *>(e->node_kids),
                  static_cast<void *>(e->node_parent), static_cast<void *>(e->node_out),
                  static_cast<void *>(e->node_up), static_cast<void *>(e->node_level),
                  static_cast<void *>(e->node_cell), static_cast<void *>(e->nexit),
                  static_cast<void *>(e->tile_n0), static_cast<void *>(e->node_tier),
                  static_cast<void *>(e->cells_list), static_cast<void *>(e->thist),
                  static_cast<void *>(e->tcur), static_cast<void *>(e->tstat)})
    if (p) (void)hipFree(p);
  if (e->graph_n_h) (void)hipHostFree(e->graph_n_h);
  for (auto &ev : e->ev)
    if (ev) (void)hipEventDestroy(ev);
  if (e->listed) (void)hipEventDestroy(e->listed);
  if (e->stream) (void)hipStreamDestroy(e->stream);
  delete e;
}

int check_ensemble(fs_ensemble *e) {
  if (!e) return FS_ERR_INVALID_ARGUMENT;
  if (e->broken) {
    fs::set_last_error("ensemble is unusable after an earlier device error");
    return FS_ERR_INTERNAL;
  }
  FS_HIP_TRY(hipSetDevice(e->device));
  return FS_OK;
}

int check_schedule(const fs_schedule &s) {
  if (s.recv_rows < kRecvRows || s.recv_rows > 256 || s.recv_rows % kRecvRows != 0 ||
      s.tiles_per_claim < 1 || s.tiles_per_claim > 16 || s.group_cells < 0)
    return FS_ERR_INVALID_ARGUMENT;
  return FS_OK;
}

// The tile-graph step of the realizations k_ens_lists listed as deep
// (fs_deep.h), on the same stream.  The host reads the list's tile count
// (one wait per step, while the erosion runs) so every per-tile kernel is
// launched with exactly one workgroup per tile.
template <int NM, bool kChain>
int graph_launches(fs_ensemble *e, const deep::GraphWork &w, int T) {
  hipStream_t s = e->stream;
  const double *h_old = e->h[e->cur];
  double *h_new = e->h[e->cur ^ 1];
  hipLaunchKernelGGL(deep::k_deep_local, dim3(T), dim3(deep::kLocalBlock), 0, s, w, e->rcv, e->cnt,
                     e->dinfo, e->link, e->node_word, e->node_kids, e->node_cell, e->nexit,
                     e->tile_n0, e->cells_list, h_new, e->tstat);
  hipLaunchKernelGGL(deep::k_deep_links, dim3(T), dim3(deep::kNodeCap), 0, s, w, e->rcv, e->link,
                     e->dinfo, e->node_cell, e->nexit, e->tile_n0, e->node_parent, e->node_kids,
                     e->node_up, e->tstat);
  hipLaunchKernelGGL(deep::k_deep_nodes, dim3(2 * T), dim3(deep::kNodeCap), 0, s, w,
                     e->node_parent, e->nexit, e->node_tier, e->node_up, e->node_level, e->thist,
                     e->tcur, e->graph_queues, e->node_word, e->node_kids, e->node_out, e->tstat);
  hipLaunchKernelGGL(deep::k_deep_levels, dim3(T), dim3(deep::kBlock), 0, s, w, e->dinfo, e->link,
                     e->node_level);
  hipLaunchKernelGGL((deep::k_deep_counts<NM, kChain>), dim3(T), dim3(deep::kCntBlock), 0, s, w, e->rcv,
                     e->cnt, e->dinfo, e->link, e->node_out, e->node_cell, e->node_tier, e->nexit,
                     e->tile_n0, e->cells_list, e->tcur, e->items, e->ftab, h_old, h_new);
  hipLaunchKernelGGL(deep::k_deep_erode<NM>, dim3(static_cast<unsigned>(e->graph_blocks)),
                     dim3(deep::kEroBlock), 0, s, w, e->rcv, e->cnt, e->cells_list, e->items,
                     e->ftab, h_old, h_new, e->tstat, e->graph_queues);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    fs::set_last_error(std::string("tile-graph launch: ") + hipGetErrorString(err));
    return FS_ERR_HIP;
  }
  return FS_OK;
}

int graph_step(fs_ensemble *e) {
  FS_HIP_TRY(hipEventSynchronize(e->listed));
  const int T = e->graph_n_h[1];
  if (T <= 0) return FS_OK;
  deep::GraphWork w;
  w.grid = e->graph_grid;
  w.first = e->tabG_off;
  w.which = e->tabG_real;
  w.size = e->tabG_size;
  e->graph_tiles += static_cast<uint64_t>(T);
  if (e->nm_all == 1) return graph_launches<1, false>(e, w, T);
  const bool chain = deep::counts_chain(T, e->ncu);
  if (e->nm_all == 2)
    return chain ? graph_launches<2, true>(e, w, T) : graph_launches<2, false>(e, w, T);
  return chain ? graph_launches<-1, true>(e, w, T) : graph_launches<-1, false>(e, w, T);
}

// A grid of at least n workgroups (a grid of one row holds fewer than 2^32
// threads).
dim3 ens_grid(int n) {
  const unsigned x = std::min(static_cast<unsigned>(n), 1u << 20);
  return dim3(x, (static_cast<unsigned>(n) + x - 1) / x);
}

template <int NM>
void launch_ens_erode(fs_ensemble *e, const EnsArgs &a) {
  const int per = e->sched.tiles_per_claim;
  const dim3 grid = ens_grid((e->tiles - 1) / per + 1);
  if (per > 1)
    hipLaunchKernelGGL((k_ens_erode<NM, true>), grid, dim3(kEroBlock), 0, e->stream, a,
                       e->tile_real, e->tiles, per);
  else
    hipLaunchKernelGGL((k_ens_erode<NM, false>), grid, dim3(kEroBlock), 0, e->stream, a,
                       e->tile_real, e->tiles, per);
}

int tile_launches(fs_ensemble *e) {
  hipStream_t s = e->stream;
  EnsArgs a{};
  a.real = e->real_d;
  a.R = e->R;
  a.h_old = e->h[e->cur];
  a.h_new = e->h[e->cur ^ 1];
  a.rcv = e->rcv;
  a.lvl = e->lvl;
  a.cnt = e->cnt;
  a.plan = e->plan;
  a.ftab = e->ftab;
  a.rh = e->rh;
  a.hist = e->hist;
  const int recv = std::max(1, e->sched.recv_rows / kRecvPerBlock);
  const dim3 recv_grid = ens_grid((e->recv_blocks - 1) / recv + 1);
  if (recv > 1)
    hipLaunchKernelGGL(k_ens_receivers<true>, recv_grid, dim3(256), 0, s, a, e->recv_real,
                       e->recv_blocks, recv);
  else
    hipLaunchKernelGGL(k_ens_receivers<false>, recv_grid, dim3(256), 0, s, a, e->recv_real,
                       e->recv_blocks, recv);
  // as for one grid: 1024-thread workgroups where there are fewer tiles than
  // four per CU
  if (e->tiles < 4 * e->ncu)
    hipLaunchKernelGGL(k_ens_acc<kAccBlockWide>, ens_grid(e->tiles), dim3(kAccBlockWide), 0, s, a,
                       e->tile_real, e->tiles);
  else
    hipLaunchKernelGGL(k_ens_acc<kAccBlock>, ens_grid(e->tiles), dim3(kAccBlock), 0, s, a,
                       e->tile_real, e->tiles);
  hipLaunchKernelGGL(k_ens_lists, dim3(1), dim3(kEnsBlock), 0, s, a, e->tabG_off, e->tabG_real,
                     e->tabG_size, e->graph_n_h);
  FS_HIP_TRY(hipEventRecord(e->listed, s));
  if (e->nm_all == 1) launch_ens_erode<1>(e, a);
  else if (e->nm_all == 2) launch_ens_erode<2>(e, a);
  else launch_ens_erode<-1>(e, a);
  FS_HIP_TRY(hipGetLastError());
  return FS_OK;
}

int launch_step(fs_ensemble *e) {
  int st = tile_launches(e);
  if (st == FS_OK) st = graph_step(e);
  if (st != FS_OK) {
    e->broken = true;
    return st;
  }
  e->cur ^= 1;
  e->steps++;
  e->have_step = true;
  return FS_OK;
}

// Device error bits of every realization, after a sync.
int ensemble_errors(fs_ensemble *e) {
  FS_HIP_TRY(hipStreamSynchronize(e->stream));
  int32_t ts[deep::kStWords];
  FS_HIP_TRY(hipMemcpy(ts, e->tstat, sizeof(ts), hipMemcpyDeviceToHost));
  if (ts[deep::kStErr]) {
    e->broken = true;
    fs::set_last_error(ts[deep::kStErr] & deep::kErrTier
                           ? "tile-graph step: a drainage path crosses more tile borders than levels allow"
                       : ts[deep::kStErr] & deep::kErrCount
                           ? "tile-graph step: work items were not all counted"
                           : "tile-graph step: receivers do not form a forest");
    return ts[deep::kStErr] & deep::kErrTier ? FS_ERR_LEVEL_OVERFLOW : FS_ERR_INTERNAL;
  }
  std::vector<int32_t> rh(static_cast<size_t>(e->R) * kRH);
  FS_HIP_TRY(hipMemcpy(rh.data(), e->rh, rh.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
  for (int r = 0; r < e->R; r++) {
    const int32_t err = rh[static_cast<size_t>(r) * kRH + kRhErr];
    if (!err) continue;
    e->broken = true;
    fs::set_last_error("realization error flags " + std::to_string(err));
    if (err & kErrNewton) return FS_ERR_NEWTON;
    if (err & kErrDepth) return FS_ERR_LEVEL_OVERFLOW;
    return FS_ERR_INTERNAL;
  }
  return FS_OK;
}

double elapsed_ms(hipEvent_t a, hipEvent_t b) {
  float ms = 0.f;
  if (hipEventElapsedTime(&ms, a, b) != hipSuccess) return -1.0;
  return ms;
}

// Time `steps` real steps with schedule s; returns ms per step (< 0 on error).
int timed_steps(fs_ensemble *e, const fs_schedule &s, int steps, double *ms_per_step) {
  e->sched = s;
  FS_HIP_TRY(hipEventRecord(e->ev[0], e->stream));
  for (int i = 0; i < steps; i++) FS_TRY(launch_step(e));
  FS_HIP_TRY(hipEventRecord(e->ev[1], e->stream));
  FS_HIP_TRY(hipEventSynchronize(e->ev[1]));
  const double ms = elapsed_ms(e->ev[0], e->ev[1]);
  e->step_ms += ms;
  *ms_per_step = ms / steps;
  return FS_OK;
}

// Coordinate search over the schedule knobs, each candidate timed on
// tune_trial real steps; stops early when `budget` steps are used.  A candidate
// has to be ahead of the best so far by more than one step's time varies (3%),
// both as timed before it and as timed again behind it: the first steps of a run
// are its slowest, and what comes later would win by that alone.  A knob is done
// with its first value that is not ahead, since more work per workgroup then only
// costs more.  Returns the number of steps taken in *used.
int autotune(fs_ensemble *e, int budget, int *used) {
  *used = 0;
  fs_schedule best = e->sched;
  double best_ms = -1;
  bool open = true;   // steps are left
  auto trial = [&](const fs_schedule &c, double *ms) {
    open = *used + e->tune_trial <= budget;
    if (!open) return FS_OK;
    FS_TRY(timed_steps(e, c, e->tune_trial, ms));
    *used += e->tune_trial;
    e->tune_cand.push_back(c);
    e->tune_ms.push_back(*ms);
    return FS_OK;
  };
  auto search = [&](int fs_schedule::*knob, std::initializer_list<int> values) {
    for (int v : values) {
      fs_schedule c = best;
      c.*knob = v;
      if (best_ms >= 0 && c.*knob == best.*knob) continue;   // timed already
      double ms = 0, again = 0;
      FS_TRY(trial(c, &ms));
      if (!open) return FS_OK;
      if (best_ms < 0) {
        best_ms = ms;
        best = c;
        continue;
      }
      if (!(ms < 0.97 * best_ms)) return FS_OK;
      FS_TRY(trial(best, &again));
      if (!open) return FS_OK;
      best_ms = std::min(best_ms, again);
      if (!(ms < 0.97 * best_ms)) return FS_OK;
      best_ms = ms;
      best = c;
    }
    return FS_OK;
  };
  FS_TRY(search(&fs_schedule::recv_rows, {kRecvPerBlock, 2 * kRecvPerBlock, 4 * kRecvPerBlock}));
  FS_TRY(search(&fs_schedule::tiles_per_claim, {1, 2, 4}));
  e->sched = best;
  return FS_OK;
}

int run_steps(fs_ensemble *e, long long total) {
  long long done = 0;
  FS_HIP_TRY(hipEventRecord(e->ev[0], e->stream));
  bool open = true;   // ev[0] marks the start of untimed-by-tuner steps
  double plain_ms = 0;
  while (done < total) {
    const bool due = e->tune_trial > 0 &&
                     (e->tuned_at == ~0ull ||
                      (e->tune_interval > 0 && e->steps >= e->tuned_at + e->tune_interval));
    if (due) {
      if (open) {
        FS_HIP_TRY(hipEventRecord(e->ev[1], e->stream));
        FS_HIP_TRY(hipEventSynchronize(e->ev[1]));
        plain_ms += elapsed_ms(e->ev[0], e->ev[1]);
        open = false;
      }
      e->tuned_at = e->steps;
      int used = 0;
      FS_TRY(autotune(e, static_cast<int>(std::min<long long>(total - done, 1 << 30)), &used));
      done += used;
      continue;
    }
    if (!open) {
      FS_HIP_TRY(hipEventRecord(e->ev[0], e->stream));
      open = true;
    }
    FS_TRY(launch_step(e));
    done++;
  }
  if (open) {
    FS_HIP_TRY(hipEventRecord(e->ev[1], e->stream));
    FS_HIP_TRY(hipEventSynchronize(e->ev[1]));
    plain_ms += elapsed_ms(e->ev[0], e->ev[1]);
  }
  e->step_ms += plain_ms;
  return ensemble_errors(e);
}

int check_index(fs_ensemble *e, int r, size_t count, int *ri) {
  if (r < 0 || r >= e->R) return FS_ERR_INVALID_ARGUMENT;
  *ri = e->to_internal[r];
  const EnsReal &g = e->real[*ri];
  if (count != static_cast<size_t>(g.W) * g.H) return FS_ERR_BUFFER_SIZE;
  return FS_OK;
}

template <class T>
int download(fs_ensemble *e, T *dst, const T *src, size_t count) {
  FS_HIP_TRY(hipStreamSynchronize(e->stream));
  FS_HIP_TRY(hipMemcpy(dst, src, count * sizeof(T), hipMemcpyDeviceToHost));
  return FS_OK;
}

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

}  // namespace

extern "C" {

int fs_ensemble_create(const fs_realization *reals, int count, int device, fs_ensemble **out) {
  if (!out) return FS_ERR_INVALID_ARGUMENT;
  *out = nullptr;
  if (!reals || count <= 0 || count > kMaxRealizations) return FS_ERR_INVALID_ARGUMENT;
  for (int r = 0; r < count; r++) FS_TRY(fs::validate_params(reals[r].width, reals[r].height, &reals[r].params));
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0 || device < 0 || device >= ndev) {
    fs::set_last_error("no HIP device " + std::to_string(device));
    return FS_ERR_NO_DEVICE;
  }
  fs_ensemble *e = new (std::nothrow) fs_ensemble();
  if (!e) return FS_ERR_OUT_OF_MEMORY;
  struct Guard {
    fs_ensemble *e;
    ~Guard() { if (e) free_ensemble(e); }
  } guard{e};
  e->device = device;
  e->R = count;
  FS_HIP_TRY(hipSetDevice(device));
  FS_HIP_TRY(hipDeviceGetAttribute(&e->ncu, hipDeviceAttributeMultiprocessorCount, device));
  // largest realizations first
  std::vector<int> ord(count);
  std::iota(ord.begin(), ord.end(), 0);
  std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) {
    return static_cast<long long>(reals[a].width) * reals[a].height >
           static_cast<long long>(reals[b].width) * reals[b].height;
  });
  e->to_internal.resize(count);
  e->spec.resize(count);
  e->real.resize(count);
  size_t cells = 0, ftab_n = 0, lev_n = 0;
  int nm0 = -2;
  long long recv_total = 0;   // receiver workgroups
  for (int i = 0; i < count; i++) {
    const fs_realization &s = reals[ord[i]];
    e->to_internal[ord[i]] = i;
    e->spec[i] = s;
    EnsReal &g = e->real[i];
    const size_t n = static_cast<size_t>(s.width) * s.height;
    g.off = cells;
    g.W = s.width;
    g.H = s.height;
    g.tiles_x = (s.width + kTile - 1) / kTile;
    g.ntiles = g.tiles_x * ((s.height + kTile - 1) / kTile);
    g.recv_xb = (s.width - 4 + kWave - 1) / kWave;
    const int groups = (s.height - 4 + kRecvShort - 1) / kRecvShort;
    const long long blocks =
        static_cast<long long>(g.recv_xb) * ((groups + kRecvGroups - 1) / kRecvGroups);
    if (recv_total + blocks >= (1ll << 31)) return FS_ERR_DIMENSIONS;
    g.recv_first = static_cast<int>(recv_total);
    recv_total += blocks;
    g.d_card = s.params.dx;
    g.d_diag = s.params.dx * fs::kSqrt2;
    g.ek = make_erode_const(s.params, &g.nmode);
    g.ftab_off = ftab_n;
    g.lev_off = lev_n;
    g.lev_cap = static_cast<int>(std::min<size_t>(n, FS_MAX_LEVELS) + 3);
    nm0 = nm0 == -2 ? g.nmode : (nm0 == g.nmode ? nm0 : -1);
    cells += align_up(n, 64);
    ftab_n += align_up(2 * (std::max<size_t>(n, kFactCache - 1) + 1), 64);
    lev_n += align_up(static_cast<size_t>(g.lev_cap), 64);
  }
  e->nm_all = nm0 == 0 ? -1 : nm0;
  e->cells = cells;
  long long tiles_total = 0;
  for (EnsReal &g : e->real) {
    g.plan_off = static_cast<uint64_t>(tiles_total);
    tiles_total += g.ntiles;
  }
  if (tiles_total >= (1ll << 31)) return FS_ERR_DIMENSIONS;
  e->tiles = static_cast<int>(tiles_total);
  e->recv_blocks = static_cast<int>(recv_total);

  FS_HIP_TRY(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking));
  for (auto &ev : e->ev) FS_HIP_TRY(hipEventCreate(&ev));
  FS_HIP_TRY(hipEventCreateWithFlags(&e->listed, hipEventDisableTiming));
  FS_TRY(fs::dev_alloc(&e->real_d, count));
  FS_TRY(fs::dev_alloc(&e->h[0], cells));
  FS_TRY(fs::dev_alloc(&e->h[1], cells));
  FS_TRY(fs::dev_alloc(&e->rcv, cells + 16));
  FS_TRY(fs::dev_alloc(&e->lvl, cells));
  FS_TRY(fs::dev_alloc(&e->cnt, cells));
  FS_TRY(fs::dev_alloc(&e->plan, static_cast<size_t>(tiles_total)));
  FS_TRY(fs::dev_alloc(&e->lev, lev_n));
  FS_TRY(fs::dev_alloc(&e->ftab, ftab_n));
  FS_TRY(fs::dev_alloc(&e->rh, static_cast<size_t>(count) * kRH));
  FS_TRY(fs::dev_alloc(&e->hist, static_cast<size_t>(count) * kHistLen));
  FS_TRY(fs::dev_alloc(&e->recv_real, static_cast<size_t>(recv_total)));
  FS_TRY(fs::dev_alloc(&e->tile_real, static_cast<size_t>(tiles_total)));
  {
    std::vector<int32_t> of;
    try {
      of.resize(static_cast<size_t>(std::max(recv_total, tiles_total)));
    } catch (const std::bad_alloc &) {
      return FS_ERR_OUT_OF_MEMORY;
    }
    for (int r = 0; r < count; r++) {
      const EnsReal &g = e->real[r];
      const long long end = r + 1 < count ? e->real[r + 1].recv_first : recv_total;
      std::fill(of.begin() + g.recv_first, of.begin() + static_cast<std::ptrdiff_t>(end), r);
    }
    FS_HIP_TRY(hipMemcpy(e->recv_real, of.data(), static_cast<size_t>(recv_total) * sizeof(int32_t),
                         hipMemcpyHostToDevice));
    for (int r = 0; r < count; r++) {
      const EnsReal &g = e->real[r];
      std::fill_n(of.begin() + static_cast<std::ptrdiff_t>(g.plan_off), g.ntiles, r);
    }
    FS_HIP_TRY(hipMemcpy(e->tile_real, of.data(),
                         static_cast<size_t>(tiles_total) * sizeof(int32_t),
                         hipMemcpyHostToDevice));
  }
  FS_TRY(fs::dev_alloc(&e->tabG_off, count + 1));
  FS_TRY(fs::dev_alloc(&e->tabG_real, count + 1));
  FS_TRY(fs::dev_alloc(&e->tabG_size, 2));
  // the tile-graph step (deep realizations): the realizations' tiles are
  // numbered by plan_off, so the per-tile arrays cover every tile
  {
    const size_t T = static_cast<size_t>(tiles_total);
    const size_t nodes = T * deep::kNodeCap;
    const size_t tier_words = static_cast<size_t>(deep::kTierCap + 1) * deep::kShards;
    FS_TRY(fs::dev_alloc(&e->graph_grid, count));
    FS_TRY(fs::dev_alloc(&e->dinfo, cells));
    FS_TRY(fs::dev_alloc(&e->link, cells));
    FS_TRY(fs::dev_alloc(&e->node_word, nodes));
    FS_TRY(fs::dev_alloc(&e->node_kids, nodes));
    FS_TRY(fs::dev_alloc(&e->node_parent, nodes));
    FS_TRY(fs::dev_alloc(&e->node_out, nodes));
    FS_TRY(fs::dev_alloc(&e->node_up, nodes));
    FS_TRY(fs::dev_alloc(&e->node_level, nodes));
    FS_TRY(fs::dev_alloc(&e->node_cell, nodes));
    FS_TRY(fs::dev_alloc(&e->node_tier, nodes));
    FS_TRY(fs::dev_alloc(&e->nexit, T));
    FS_TRY(fs::dev_alloc(&e->tile_n0, T));
    FS_TRY(fs::dev_alloc(&e->cells_list, T * deep::kCells));
    FS_TRY(fs::dev_alloc(&e->items, T * deep::kTiersPerTile));
    FS_TRY(fs::dev_alloc(&e->thist, tier_words));
    FS_TRY(fs::dev_alloc(&e->tcur, tier_words));
    FS_TRY(fs::dev_alloc(&e->tstat, deep::kStWords));
    FS_HIP_TRY(hipMemset(e->thist, 0, tier_words * sizeof(int32_t)));
    FS_HIP_TRY(hipMemset(e->tstat, 0, deep::kStWords * sizeof(int32_t)));
    if (hipHostMalloc(reinterpret_cast<void **>(&e->graph_n_h), 2 * sizeof(int32_t)) !=
        hipSuccess) {
      e->graph_n_h = nullptr;
      fs::set_last_error("hipHostMalloc failed");
      return FS_ERR_OUT_OF_MEMORY;
    }
  }
  FS_HIP_TRY(hipMemcpy(e->real_d, e->real.data(), count * sizeof(EnsReal), hipMemcpyHostToDevice));
  {
    std::vector<deep::GraphGrid> gg(count);
    for (int r = 0; r < count; r++) {
      const EnsReal &g = e->real[r];
      deep::GraphGrid &d = gg[r];
      d.off = g.off;
      d.ftab_off = g.ftab_off;
      d.hdr = e->rh + static_cast<size_t>(r) * kRH;   // [0] depth, [2] error bits
      d.levels = e->lev + g.lev_off;
      d.W = g.W;
      d.H = g.H;
      d.tiles_x = g.tiles_x;
      d.tile0 = static_cast<int>(g.plan_off);
      d.nlev = g.lev_cap;
      d.nmode = g.nmode;
      d.ek = g.ek;
    }
    FS_HIP_TRY(hipMemcpy(e->graph_grid, gg.data(), gg.size() * sizeof(deep::GraphGrid),
                         hipMemcpyHostToDevice));
  }
  FS_HIP_TRY(hipMemset(e->rcv, 0xFF, cells + 16));   // rings never get a receiver, RB:361-362
  FS_HIP_TRY(hipMemset(e->cnt, 0, cells * sizeof(uint32_t)));
  FS_HIP_TRY(hipMemset(e->rh, 0, static_cast<size_t>(count) * kRH * sizeof(int32_t)));
  FS_HIP_TRY(hipMemset(e->hist, 0, static_cast<size_t>(count) * kHistLen * sizeof(int32_t)));

  // Initial terrains and erosion factor tables.  Host threads fill host
  // buffers, one realization each per round; this thread alone makes every
  // HIP call (no HIP state is created on threads that exit).
  unsigned nt = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
  nt = std::min<unsigned>(nt, static_cast<unsigned>(count));
  std::vector<std::vector<double>> terr(nt), tabs(nt);
  for (int r0 = 0; r0 < count; r0 += static_cast<int>(nt)) {
    const int nr = std::min(static_cast<int>(nt), count - r0);
    std::vector<int> status(static_cast<size_t>(nr), FS_OK);
    auto fill = [&](int w) {
      const int i = r0 + w;
      const EnsReal &g = e->real[i];
      const fs_realization &s = e->spec[i];
      const size_t n = static_cast<size_t>(g.W) * g.H;
      const size_t kmax = std::max<size_t>(n, kFactCache - 1);
      try {
        terr[w].resize(n);
        tabs[w].resize(2 * (kmax + 1));
      } catch (const std::bad_alloc &) {
        status[w] = FS_ERR_OUT_OF_MEMORY;
        return;
      }
      fs::generate_terrain(terr[w].data(), g.W, g.H, s.engine_seed);
      fs::fill_fact_table(tabs[w].data(), kmax, s.params.cell_area, s.params.meq, g.ek.kdt,
                          g.ek.lenpow0, g.ek.lenpow1);
    };
    {
      std::vector<std::thread> pool;
      for (int w = 1; w < nr; w++) pool.emplace_back(fill, w);
      fill(0);
      for (auto &th : pool) th.join();
    }
    for (int w = 0; w < nr; w++) {
      if (status[w] != FS_OK) {
        fs::set_last_error("initialising realizations failed");
        return status[w];
      }
      const EnsReal &g = e->real[r0 + w];
      FS_HIP_TRY(hipMemcpy(e->h[0] + g.off, terr[w].data(), terr[w].size() * sizeof(double),
                           hipMemcpyHostToDevice));
      FS_HIP_TRY(hipMemcpy(e->ftab + g.ftab_off, tabs[w].data(), tabs[w].size() * sizeof(double),
                           hipMemcpyHostToDevice));
    }
  }

  e->graph_blocks = e->nm_all == 1   ? deep::erode_grid<1>(e->ncu)
                    : e->nm_all == 2 ? deep::erode_grid<2>(e->ncu)
                                     : deep::erode_grid<-1>(e->ncu);
  e->graph_queues = deep::erode_queues(e->graph_blocks);
  FS_HIP_TRY(hipDeviceSynchronize());
  guard.e = nullptr;
  *out = e;
  return FS_OK;
}

int fs_ensemble_destroy(fs_ensemble *e) {
  if (!e) return FS_ERR_INVALID_ARGUMENT;
  free_ensemble(e);
  return FS_OK;
}

int fs_ensemble_size(fs_ensemble *e, int *count, size_t *cells) {
  if (!e) return FS_ERR_INVALID_ARGUMENT;
  if (count) *count = e->R;
  if (cells) {
    size_t c = 0;
    for (const EnsReal &g : e->real) c += static_cast<size_t>(g.W) * g.H;
    *cells = c;
  }
  return FS_OK;
}

int fs_ensemble_run(fs_ensemble *e, int nstep) {
  FS_TRY(check_ensemble(e));
  if (nstep < 0) return FS_ERR_INVALID_ARGUMENT;
  return run_steps(e, static_cast<long long>(nstep) + 1);
}

int fs_ensemble_step(fs_ensemble *e) {
  FS_TRY(check_ensemble(e));
  return run_steps(e, 1);
}

int fs_ensemble_get_h(fs_ensemble *e, int r, double *h, size_t count) {
  FS_TRY(check_ensemble(e));
  if (!h) return FS_ERR_INVALID_ARGUMENT;
  int ri;
  FS_TRY(check_index(e, r, count, &ri));
  return download(e, h, e->h[e->cur] + e->real[ri].off, count);
}

int fs_ensemble_set_h(fs_ensemble *e, int r, const double *h, size_t count) {
  FS_TRY(check_ensemble(e));
  if (!h) return FS_ERR_INVALID_ARGUMENT;
  int ri;
  FS_TRY(check_index(e, r, count, &ri));
  FS_HIP_TRY(hipStreamSynchronize(e->stream));
  FS_HIP_TRY(hipMemcpy(e->h[e->cur] + e->real[ri].off, h, count * sizeof(double),
                       hipMemcpyHostToDevice));
  return FS_OK;
}

int fs_ensemble_get_receivers(fs_ensemble *e, int r, int32_t *rec, size_t count) {
  FS_TRY(check_ensemble(e));
  if (!rec) return FS_ERR_INVALID_ARGUMENT;
  int ri;
  FS_TRY(check_index(e, r, count, &ri));
  std::vector<uint8_t> v(count);
  FS_TRY(download(e, v.data(), e->rcv + e->real[ri].off, count));
  for (size_t i = 0; i < count; i++) rec[i] = v[i] == kNoFlow ? FS_NO_FLOW : v[i];
  return FS_OK;
}

int fs_ensemble_get_accum(fs_ensemble *e, int r, double *accum, size_t count) {
  FS_TRY(check_ensemble(e));
  if (!accum) return FS_ERR_INVALID_ARGUMENT;
  int ri;
  FS_TRY(check_index(e, r, count, &ri));
  const EnsReal &g = e->real[ri];
  int32_t q[kRH];
  FS_TRY(download(e, q, e->rh + static_cast<size_t>(ri) * kRH, kRH));
  std::vector<uint32_t> v(count);
  FS_TRY(download(e, v.data(), e->cnt + g.off, count));
  const double area = e->spec[ri].params.cell_area;
  for (size_t i = 0; i < count; i++) accum[i] = static_cast<double>(v[i]) * area;
  return FS_OK;
}

int fs_ensemble_get_levels(fs_ensemble *e, int r, int32_t *levels, size_t capacity,
                           int32_t *nlevel) {
  FS_TRY(check_ensemble(e));
  if (!nlevel || r < 0 || r >= e->R) return FS_ERR_INVALID_ARGUMENT;
  *nlevel = 0;
  if (!e->have_step) return FS_OK;
  const int ri = e->to_internal[r];
  const EnsReal &g = e->real[ri];
  const int32_t n = g.W * g.H;
  int32_t q[kRH];
  FS_TRY(download(e, q, e->rh + static_cast<size_t>(ri) * kRH, kRH));
  const int D = q[kRhDepth];
  if (D < 0 || D + 3 > g.lev_cap) return FS_ERR_INTERNAL;
  std::vector<int32_t> lv(D + 3);
  if (q[kRhPath] == 3) {
    // the tile-graph step counted cells per level
    std::vector<int32_t> c(D + 1);
    FS_TRY(download(e, c.data(), e->lev + g.lev_off, c.size()));
    lv[0] = 0;
    for (int l = 0; l <= D; l++) lv[l + 1] = lv[l] + c[l];
    lv[D + 2] = n;
  } else {
    int32_t hist[kHistLen];
    FS_TRY(download(e, hist, e->hist + static_cast<size_t>(ri) * kHistLen, kHistLen));
    if (D >= kHistLen) return FS_ERR_INTERNAL;
    lv[0] = 0;
    for (int l = 0; l <= D; l++) lv[l + 1] = lv[l] + hist[l];
    lv[D + 2] = n;
  }
  if (lv[D + 1] != n) {
    fs::set_last_error("level sizes cover " + std::to_string(lv[D + 1]) + " of " +
                       std::to_string(n) + " cells");
    return FS_ERR_INTERNAL;
  }
  *nlevel = D + 3;
  if (!levels) return FS_OK;
  if (capacity < static_cast<size_t>(*nlevel)) return FS_ERR_BUFFER_SIZE;
  std::copy(lv.begin(), lv.end(), levels);
  return FS_OK;
}

int fs_ensemble_path_stats(fs_ensemble *e, int r, uint64_t *tile_steps, uint64_t *level_steps) {
  FS_TRY(check_ensemble(e));
  if (r < 0 || r >= e->R) return FS_ERR_INVALID_ARGUMENT;
  int32_t q[kRH];
  FS_TRY(download(e, q, e->rh + static_cast<size_t>(e->to_internal[r]) * kRH, kRH));
  if (tile_steps) *tile_steps = static_cast<uint32_t>(q[kRhTileSteps]);
  if (level_steps) *level_steps = static_cast<uint32_t>(q[kRhLevelSteps]);
  return FS_OK;
}

int fs_ensemble_set_schedule(fs_ensemble *e, const fs_schedule *s) {
  FS_TRY(check_ensemble(e));
  if (!s) return FS_ERR_INVALID_ARGUMENT;
  FS_TRY(check_schedule(*s));
  e->sched = *s;
  return FS_OK;
}

int fs_ensemble_get_schedule(fs_ensemble *e, fs_schedule *s) {
  if (!e || !s) return FS_ERR_INVALID_ARGUMENT;
  *s = e->sched;
  return FS_OK;
}

int fs_ensemble_autotune(fs_ensemble *e, int trial_steps, int interval) {
  FS_TRY(check_ensemble(e));
  if (trial_steps < 0 || interval < 0) return FS_ERR_INVALID_ARGUMENT;
  e->tune_trial = trial_steps;
  e->tune_interval = interval;
  e->tuned_at = ~0ull;
  return FS_OK;
}

int fs_ensemble_tune_log(fs_ensemble *e, fs_schedule *cand, double *ms_per_step, int capacity,
                         int *count) {
  if (!e || !count) return FS_ERR_INVALID_ARGUMENT;
  *count = static_cast<int>(e->tune_cand.size());
  if (!cand && !ms_per_step) return FS_OK;
  if (capacity < *count) return FS_ERR_BUFFER_SIZE;
  for (int i = 0; i < *count; i++) {
    if (cand) cand[i] = e->tune_cand[i];
    if (ms_per_step) ms_per_step[i] = e->tune_ms[i];
  }
  return FS_OK;
}

int fs_ensemble_stats(fs_ensemble *e, uint64_t *steps, double *step_ms) {
  if (!e) return FS_ERR_INVALID_ARGUMENT;
  if (steps) *steps = e->steps;
  if (step_ms) *step_ms = e->step_ms;
  return FS_OK;
}

int fs_ensemble_synchronize(fs_ensemble *e) {
  FS_TRY(check_ensemble(e));
  FS_HIP_TRY(hipStreamSynchronize(e->stream));
  return FS_OK;
}

}  // extern "C"
