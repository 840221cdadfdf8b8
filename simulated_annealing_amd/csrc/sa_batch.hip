// sa_batch.hip -- many independent instances of uneven size swept together (the
// C ABI sa_batch_* of include/sa_hip.h).
//
// Each instance is a ladder (couplings, spins, nsys systems) with its own counter
// RNG seed and either an anneal (temperatures per sweep) or parallel tempering
// (fixed ladder of temperatures, an exchange attempt every `every` sweeps).
//
// Sweeps.  A half-sweep launch covers every unfinished instance.  The work items
// (3D: (column, system), 2D: (site, system)) of all instances are cut into blocks
// of one instance each; the block map and the per-instance descriptors live in
// device memory and a fixed grid walks the block map (grid-stride), so the launch
// sequence of a chunk of sweeps does not depend on which instances are present: it
// is captured once per chunk length as a hipGraph and replayed while instances
// come and go.  Every block runs the per-column / per-site code of the
// single-instance kernels, so an instance's spins are bit for bit those of its
// ladder swept alone.  The descriptors hold each instance's sweep index at the
// start of the chunk; every launch of the chunk gets its sweep's offset as a
// constant argument, and one one-block kernel at the end of the chunk advances the
// indices (no index update, and no drain of the whole grid for one, per sweep).
//
// Tiles.  Instances with symmetric tables that fit take the LDS-resident sweeps of
// sa_tile2d.hpp / sa_tile3d.hpp instead: 3D instances tiles of columns, one launch per
// sweep for all of them, 2D ones with an even side the whole lattice or bands of rows, one
// launch per four sweeps.  They need a second
// spin array (tiles and bands read one and write the other) and, in 3D, the couplings with
// z fastest; where that memory is not to be had, an instance takes the half-sweep kernels.
//
// Exchanges.  Chunks end on every parallel-tempering instance's exchange points.
// There the host draws the pair and the uniform of each due instance (its own
// mt19937(123), as parallel_tempering::step), one launch measures the coldest
// system and the pair of all due instances, the host decides the lane masks with
// the reference's rule, and one launch applies all masked swaps.
//
// Tuning.  Threads per block and sweeps per graph are picked online: the first
// chunks try the candidates (results do not depend on them), the fastest per work
// item is kept.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <memory>
#include <vector>

#include "sa/exchange.hpp"
#include "sa_internal.hpp"
#include "sa_per_device.hpp"
#include "sa_tile2d.hpp"
#include "sa_tile3d.hpp"

namespace {

// how an instance is swept
enum { FORM_HALF = 0, FORM_3D = 1, FORM_3D_ODD = 2, FORM_2D_WHOLE = 3, FORM_2D_BANDS = 4 };
__host__ __device__ __forceinline__ bool two_arrays(int form) {
  return form == FORM_3D || form == FORM_3D_ODD || form == FORM_2D_BANDS;
}

struct inst_desc {
  sa::sweep_args a;  // a.s: current spin array at the schedule; tab: tables (per sweep: nsweeps x nsys, else nsys)
  uint64_t *s2;      // second spin array (forms with two arrays)
  int kind, nsweeps, t, per_sweep, fast;
  int form;
  int cur;           // 1: s2 holds the current spins
  int m;             // sweeps of one visit (forms 3D: 1)
  int th, bands;     // 2D forms
  sa::tile3d_args t3;  // 3D forms: geometry and couplings
};

// t: the instance's sweep index (its index at the chunk start plus the sweep's
// offset in the chunk, a constant of the captured launch)
template <bool FAST>
__device__ __forceinline__ void batch_item(const inst_desc &in, int t, int color, int k, int sys) {
  sa::sweep_args a = in.a;
  if (in.per_sweep) a.tab += (int64_t)t * a.nsys;
  a.sweep = (uint64_t)t;
  if (a.L & 1) {  // odd L: k is a member lane (3D) or a wrap group (2D), sa_kernels.hpp
    if (in.kind == SA_KIND_3D) sa::odd3d_lane<true, FAST>(a, color, k, sys);
    else if (in.kind == SA_KIND_2D) sa::odd2d_group<true, FAST, false>(a, color, k, sys);
    else sa::odd2d_group<true, false, true>(a, color, k, sys);
    return;
  }
  if (in.kind == SA_KIND_3D) sa::half3d_column<true, FAST, 1, true>(a, color, k, sys);
  else if (in.kind == SA_KIND_2D) sa::half2d_site<true, FAST, false, 1>(a, color, k, sys);
  else sa::half2d_site<true, false, true, 1>(a, color, k, sys);
}

// work items of one system in a half-sweep: columns (3D) or sites (2D) of one
// colour for even L; for odd L the member lanes (3D, a multiple of 64 so that each
// system starts at a wave boundary) or the wrap groups (2D)
__host__ __device__ __forceinline__ int half_items(int kind, int L) {
  if (!(L & 1)) return L * (L >> 1);
  return kind == SA_KIND_3D ? sa::odd_width(L) : sa::odd_groups(L);
}

// ctrl[0] = blocks in the block map, ctrl[1] = descriptors; s = the sweep's offset in
// the chunk (descriptors hold the sweep index at the chunk start)
__global__ void __launch_bounds__(256) k_batch_half(const inst_desc *__restrict__ d, const int2 *__restrict__ bmap,
                                                    const int *__restrict__ ctrl, int color, int s) {
  const int nb = ctrl[0];
  for (int blk = blockIdx.x; blk < nb; blk += gridDim.x) {
    const int2 bm = bmap[blk];
    const inst_desc &in = d[bm.x];
    const int t = in.t + s;
    if (t >= in.nsweeps) continue;
    const int work = half_items(in.kind, in.a.L);
    const int item = bm.y + (int)threadIdx.x;
    if (item >= work * in.a.nsys) continue;
    const int sys = item / work, k = item - sys * work;
    if (in.fast) batch_item<true>(in, t, color, k, sys);
    else batch_item<false>(in, t, color, k, sys);
  }
}

// end of a chunk of k sweeps: sweep indices advance by the sweeps each instance did
__global__ void k_batch_advance(inst_desc *d, const int *__restrict__ ctrl, int k) {
  const int n = ctrl[1];
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int done = min(k, max(0, d[i].nsweeps - d[i].t));
    d[i].t += done;
    if (two_arrays(d[i].form)) d[i].cur ^= ((done + d[i].m - 1) / d[i].m) & 1;  // each visit wrote the other array
  }
}

// Launch v of a chunk of k sweeps: sweeps v*m .. of every listed tile, at most m of them.
// Returns false when the instance has none left; a.s and out are the arrays of this launch.
__device__ __forceinline__ bool tile_visit(const inst_desc &in, int k, int v, sa::sweep_args &a, uint64_t *&out, int &ns) {
  const int t = in.t + v * in.m;
  ns = min(in.m, min(in.nsweeps - t, k - v * in.m));
  if (ns <= 0) return false;
  const int cur = two_arrays(in.form) ? in.cur ^ (v & 1) : 0;
  a = in.a;
  if (in.per_sweep) a.tab += (int64_t)t * a.nsys;
  a.sweep = (uint64_t)t;
  a.s = cur ? in.s2 : in.a.s;
  out = cur ? in.a.s : in.s2;
  return true;
}

// The 3D tiles of a sweep.  Entries (descriptor, tile) are kept per XCD (blocks go
// round-robin over the 8 XCDs), an instance's tiles together, so its words and couplings
// stay in one L2: ctrl[2+2x], ctrl[3+2x] = first entry and count of XCD x.
// Blocks of 512 threads with 80 KB of LDS: two per CU, eight waves each.
// 13 systems of L=48: 55 -> 22 us per sweep, of L=47 77 -> 25, of L=24 25 -> 8 (column walks
// in two launches before); segments of four planes take the same.  In one kernel with the 2D
// tiles the registers spilled and the two kinds' blocks waited for each other (the benchmark
// mix 73 us per sweep against 52).
constexpr int kTileThreads = 512, kTileS = 2;
constexpr size_t kTileLds = 80 * 1024;
__global__ void __launch_bounds__(kTileThreads, 4) k_batch_tile3d(const inst_desc *__restrict__ d,
                                                                  const int2 *__restrict__ tmap,
                                                                  const int *__restrict__ ctrl, int k, int v) {
  extern __shared__ __align__(16) uint64_t lds[];
  const int xcd = (int)blockIdx.x & 7, off = ctrl[2 + 2 * xcd], n = ctrl[3 + 2 * xcd];
  for (int e = (int)blockIdx.x >> 3; e < n; e += (int)gridDim.x >> 3) {  // the same for the whole block
    const int2 tm = tmap[off + e];
    const inst_desc &in = d[tm.x];
    sa::tile3d_args t3 = in.t3;
    int ns;
    if (!tile_visit(in, k, v, t3.a, t3.out, ns)) continue;
    const int per = t3.ntx * t3.nty, sys = tm.y / per, r = tm.y - sys * per, by = r / t3.ntx;
    if (in.form == FORM_3D) sa::tile3d<true, true, kTileS, false, false>(t3, sys, r - by * t3.ntx, by, lds);
    else sa::tile3d_odd<true, true, kTileS, false>(t3, sys, r - by * t3.ntx, by, lds);
    __syncthreads();  // the next tile reuses the LDS
  }
}

// The 2D tiles: whole lattices and bands of rows, up to m sweeps per launch (16 systems of
// L=64: 8.1 -> 3.9 us per sweep, of L=128 10.1 -> 4.2).
constexpr int kTile2dThreads = 1024, kTile2dItems = 2 * kTile2dThreads;
constexpr int kSweeps2d = 4;  // sweeps per launch
__global__ void __launch_bounds__(kTile2dThreads) k_batch_tile2d(const inst_desc *__restrict__ d,
                                                                 const int2 *__restrict__ tmap,
                                                                 const int *__restrict__ ctrl, int k, int v) {
  extern __shared__ __align__(16) uint64_t lds[];
  const int off = ctrl[18], n = ctrl[19];
  for (int e = (int)blockIdx.x; e < n; e += (int)gridDim.x) {
    const int2 tm = tmap[off + e];
    const inst_desc &in = d[tm.x];
    sa::tile2d_args t2;
    if (!tile_visit(in, k, v, t2.a, t2.out, t2.ns)) continue;
    t2.th = in.th;
    t2.bands = in.bands;
    t2.tab_step = in.per_sweep ? t2.a.nsys : 0;
    const int sys = tm.y / in.bands;
    if (in.form == FORM_2D_WHOLE) sa::tile2d<true, sa::T2_FAST, 2, true>(t2, sys, 0, lds);
    else sa::tile2d<true, sa::T2_FAST, 2, false>(t2, sys, tm.y - sys * in.bands, lds);
    __syncthreads();  // the next tile reuses the LDS
  }
}

// ---- measurement of listed systems of many instances
// An item is up to kMeasSites consecutive sites of one system (one block of 256
// threads: 4 waves x 16 groups of 64 sites); counts go to cnt[slot*128 + lane]
// (satisfied -x,-y[,-z] bonds) and cnt[slot*128 + 64 + lane] (set spins), as in
// the single-ladder measurement.
constexpr int kMeasSites = 4096;
struct meas_item {
  const uint64_t *s, *jx, *jy, *jz;
  int64_t N, begin;
  int kind, L, slot, pad;
};

template <int KIND>
__device__ __forceinline__ void measure_item(const meas_item &it, int lane, int wv, int &sat, int &up) {
  uint64_t e[6] = {0, 0, 0, 0, 0, 0}, mc[5] = {0, 0, 0, 0, 0};
  const int64_t L = it.L, L2 = L * L, N = it.N;
  // wave wv takes groups wv, wv+4, ... (16 groups): E <= 48 < 64, M <= 16 < 32
  for (int g = wv; g < kMeasSites / 64; g += 4) {
    const int64_t i = it.begin + (int64_t)g * 64 + lane;
    uint64_t w = 0, bw = 0, bn = 0, bu = 0;
    if (i < N) {
      const int64_t x = i % L, y = (i / L) % L, z = i / L2;
      const int64_t iw = i - x + (x == 0 ? L - 1 : x - 1);
      const int64_t inn = (y == 0) ? i + L2 - L : i - L;
      w = it.s[i];
      bw = (KIND == sa::KIND_2P && x == 0) ? 0 : (it.jx[i] ^ w ^ it.s[iw]);
      bn = it.jy[i] ^ w ^ it.s[inn];
      if (KIND == sa::KIND_3D) {
        const int64_t iu = (z == 0) ? i + N - L2 : i - L2;
        bu = it.jz[i] ^ w ^ it.s[iu];
      }
    }
    const uint64_t sb = bw ^ bn ^ bu, cb = sa::maj3(bw, bn, bu);
    uint64_t t = e[0] & sb;
    e[0] ^= sb;
    uint64_t u = sa::maj3(e[1], cb, t);
    e[1] ^= cb ^ t;
#pragma unroll
    for (int b = 2; b < 6; ++b) {
      const uint64_t v = e[b] & u;
      e[b] ^= u;
      u = v;
    }
    t = w;
#pragma unroll
    for (int b = 0; b < 5; ++b) {
      const uint64_t v = mc[b] & t;
      mc[b] ^= t;
      t = v;
    }
  }
  sat = up = 0;
#pragma unroll
  for (int b = 0; b < 6; ++b) sat += __popcll(sa::wave_transpose64(e[b], lane)) << b;
#pragma unroll
  for (int b = 0; b < 5; ++b) up += __popcll(sa::wave_transpose64(mc[b], lane)) << b;
}

__global__ void __launch_bounds__(256) k_batch_measure(const meas_item *__restrict__ items, int *cnt) {
  __shared__ int red[2][64];
  const meas_item it = items[blockIdx.x];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (threadIdx.x < 128) (&red[0][0])[threadIdx.x] = 0;
  __syncthreads();
  int sat = 0, up = 0;
  if (it.kind == SA_KIND_3D) measure_item<sa::KIND_3D>(it, lane, wv, sat, up);
  else if (it.kind == SA_KIND_2D) measure_item<sa::KIND_2D>(it, lane, wv, sat, up);
  else measure_item<sa::KIND_2P>(it, lane, wv, sat, up);
  atomicAdd(&red[0][lane], sat);
  atomicAdd(&red[1][lane], up);
  __syncthreads();
  if (threadIdx.x < 128) atomicAdd(&cnt[it.slot * 128 + threadIdx.x], (&red[0][0])[threadIdx.x]);
}

// ---- masked swaps of many pairs: a ^= (a^b)&m, b ^= (a^b)&m (src/device.cuh:18-23)
constexpr int kSwapWords = 4096;
struct swap_item {
  uint64_t *a, *b;
  uint64_t mask;
  int64_t begin, end;
};

__global__ void __launch_bounds__(256) k_batch_swap(const swap_item *__restrict__ items) {
  const swap_item it = items[blockIdx.x];
  for (int64_t i = it.begin + threadIdx.x; i < it.end; i += blockDim.x) {
    const uint64_t x = it.a[i], y = it.b[i];
    const uint64_t d = (x ^ y) & it.mask;
    it.a[i] = x ^ d;
    it.b[i] = y ^ d;
  }
}

// pinned host staging that grows on demand (contents are not kept)
struct pinned {
  void *p = nullptr;
  size_t cap = 0;
  ~pinned() {
    if (p) (void)hipHostFree(p);
  }
  bool ensure(size_t bytes) {
    if (bytes <= cap) return true;
    if (p) (void)hipHostFree(p);
    p = nullptr;
    cap = 0;
    const size_t want = std::max<size_t>(bytes * 2, 4096);
    if (hipHostMalloc(&p, want, hipHostMallocDefault) != hipSuccess) {
      p = nullptr;
      return false;
    }
    cap = want;
    return true;
  }
};

// device array that grows on demand (contents are not kept)
template <class T>
struct dev_array {
  T *p = nullptr;
  size_t cap = 0;
  ~dev_array() {
    if (p) (void)hipFree(p);
  }
  // `moved`: the array has a new address (graphs that name it are stale)
  int ensure(size_t n, bool &moved) {
    moved = false;
    if (n <= cap) return SA_OK;
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    const size_t want = std::max<size_t>(n * 2, 64);
    if (hipMalloc(&p, want * sizeof(T)) != hipSuccess) {
      p = nullptr;
      return sa_fail(SA_ERR_NOMEM, "batch device array of %zu bytes", want * sizeof(T));
    }
    cap = want;
    moved = true;
    return SA_OK;
  }
};

struct pt_state {
  int every = 0;  // exchange every `every` sweeps; 0 = anneal instance
  std::vector<double> T;
  double h = 0;
  sa::mt19937 gen{};
  int uni_b = 0;
  int pend_i = 0;
  double pend_u = 0;
  std::vector<int32_t> pairs;
  std::vector<double> us;
  std::vector<uint64_t> masks;
  std::vector<float> E_min;
  std::vector<double> acc_sum;
  std::vector<int64_t> acc_n;
};

struct batch_inst {
  sa_ladder *lad = nullptr;
  sa::sys_table *tabs = nullptr;
  int nsweeps = 0, per_sweep = 0, t = 0;
  bool fast = true, live = false;
  bool lent = false;  // its ladder was handed out (sa_batch_ladder)
  int64_t work = 0;   // work items per half-sweep (all systems)
  int64_t bytes = 0;  // device memory held
  int form = FORM_HALF;
  pt_state pt;
};

// online-tuning candidates (threads per half-sweep block, sweeps per graph); the first
// chunks try them in this order
struct tune_cand {
  int block, chunk;
};
const tune_cand kCands[2] = {{128, 32}, {64, 32}};
const int kNumCands = 2;

}  // namespace

struct sa_batch {
  hipStream_t stream = nullptr;
  int device = 0, cus = 256;
  std::vector<batch_inst> inst;  // indexed by id
  // device state of the current schedule
  dev_array<inst_desc> d_desc;
  dev_array<int2> d_bmap;
  dev_array<int> d_ctrl;
  int ndesc = 0, nblocks = 0, bmap_bs = 0;
  std::vector<int> desc_id;  // instance id of each descriptor
  std::vector<int> desc_m;   // sweeps per visit of each descriptor, 0 with one array
  dev_array<int2> d_tmap;
  int ntiles = 0, ntiles2 = 0;  // entries of k_batch_tile3d, k_batch_tile2d
  bool dirty = true;
  // (chunk length, which kernels it launches) -> graph over the current arrays and block size
  std::map<std::pair<int, int>, hipGraphExec_t> graphs;
  int graph_bs = 0;
  // exchange staging
  pinned h_stage;
  dev_array<meas_item> d_meas;
  dev_array<swap_item> d_swap;
  dev_array<int> d_cnt;
  pinned h_cnt;
  // tuning: 0 = automatic
  int block = 0, chunk = 0;
  int tuned_block = 0, tuned_chunk = 0;
  std::vector<std::pair<int, float>> trials;  // (candidate, ms per work item)
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  int64_t bytes_live = 0;
};

namespace {

void drop_graphs(sa_batch *b) {
  for (auto &g : b->graphs) (void)hipGraphExecDestroy(g.second);
  b->graphs.clear();
}

int check_id(const sa_batch *b, int id) {
  if (!b) return sa_fail(SA_ERR_ARG, "null batch");
  if (id < 0 || id >= (int)b->inst.size() || !b->inst[id].live) return sa_fail(SA_ERR_ARG, "unknown instance %d", id);
  return SA_OK;
}

int grid_for(const sa_batch *b, int bs) {
  // two blocks per wave slot at 4 waves/SIMD (the sweep kernel's register
  // budget): every CU filled, few enough blocks to loop
  return std::max(1, b->cus * 16 * 2 / (bs / 64));
}

// The form an instance with symmetric tables can take: 3D tiles for 8 <= L <= 128 (from 9
// where L is odd: a tile is at least 4 columns and its halos wide), 2D with an even L up to
// 256 (a band of 2048 items then holds four sweeps' halos and 16 rows).
int tile_form(int kind, int L) {
  if (kind == SA_KIND_3D) return L < 8 || L > 128 ? FORM_HALF : (L & 1) ? FORM_3D_ODD : FORM_3D;
  if (kind != SA_KIND_2D || (L & 1) || L > 256) return FORM_HALF;
  return L * sa::tile2d_groups(L) <= kTile2dItems ? FORM_2D_WHOLE : FORM_2D_BANDS;
}

// device bytes the form needs beside the instance's own
int64_t form_bytes(int kind, int L, int nsys, int form) {
  const int64_t L2 = (int64_t)L * L, N = L2 * (kind == SA_KIND_3D ? L : 1);
  return (two_arrays(form) ? nsys * N * 8 : 0) + (kind == SA_KIND_3D && form ? 3 * L2 * sa::column_stride(L) * 8 : 0);
}

// 3D tile geometry: wide x high columns, halved until the LDS holds it
bool tile3d_geometry(sa::tile3d_args &a, int L, int wide, int high) {
  for (;;) {
    const size_t lds = sa::tile3d_setup(a, L, false, wide, high, kTileS, kTileThreads);
    if (lds && lds <= kTileLds) return true;
    if (wide <= 4 && high <= 4) return false;
    if (wide >= high) wide /= 2;
    else high /= 2;
  }
}

bool tiles_3d(int form) { return form == FORM_3D || form == FORM_3D_ODD; }

// descriptors, the half-sweep block map and the tiles of the unfinished instances,
// largest remaining work first
int rebuild(sa_batch *b, int bs) {
  // 3D tiles read a copy of the couplings: made again where the ladder was given others
  for (batch_inst &in : b->inst)
    if (in.live && in.t < in.nsweeps && tiles_3d(in.form) && !in.lad->jt_current) {
      if (!sa_detail::tile3d_couplings(in.lad)) in.form = FORM_HALF;
      SA_HIP_TRY(hipGetLastError());
      SA_HIP_TRY(hipStreamSynchronize(in.lad->stream));
    }
  std::vector<int> ids;
  for (int i = 0; i < (int)b->inst.size(); ++i)
    if (b->inst[i].live && b->inst[i].t < b->inst[i].nsweeps) ids.push_back(i);
  std::stable_sort(ids.begin(), ids.end(), [&](int x, int y) {
    const auto &a = b->inst[x], &c = b->inst[y];
    return a.work * (int64_t)(a.nsweeps - a.t) > c.work * (int64_t)(c.nsweeps - c.t);
  });
  // 3D tiles of 8 x 8 columns when they make two blocks per CU, else smaller ones
  int64_t tiles8 = 0;
  for (int id : ids) {
    const batch_inst &in = b->inst[id];
    const int64_t side = (in.lad->L + 7) / 8;
    if (tiles_3d(in.form)) tiles8 += side * side * in.lad->nsys;
  }
  const int wide = tiles8 >= 2 * b->cus / 4 ? 8 : 4, high = tiles8 >= 2 * b->cus / 2 ? 8 : 4;
  std::vector<inst_desc> descs(ids.size());
  struct item {
    int2 e;
    float cost;
  };
  std::vector<item> tiles;
  std::vector<int2> halves, tiles2;
  double total = 0;
  b->desc_m.assign(ids.size(), 0);
  for (size_t q = 0; q < ids.size(); ++q) {
    const batch_inst &in = b->inst[ids[q]];
    const sa_ladder *l = in.lad;
    inst_desc &d = descs[q];
    std::memset(&d, 0, sizeof d);
    d.a.s = l->s;  // the current array
    d.s2 = l->s_alt;
    d.a.jx = l->jx;
    d.a.jy = l->jy;
    d.a.jz = l->jz;
    d.a.tab = in.tabs;
    d.a.seed = l->seed;
    d.a.N = l->N;
    d.a.L = l->L;
    d.a.nsys = l->nsys;
    d.kind = l->kind;
    d.nsweeps = in.nsweeps;
    d.t = in.t;
    d.per_sweep = in.per_sweep;
    d.fast = in.fast ? 1 : 0;
    d.form = in.form;
    d.m = 1;
    int64_t n = 0;
    float cost = 0;  // of an entry, about us
    if (tiles_3d(in.form) && tile3d_geometry(d.t3, l->L, wide, high)) {
      const int64_t jn = (int64_t)l->L * l->L * sa::column_stride(l->L);
      d.t3.jxt = l->jt;
      d.t3.jyt = l->jt + jn;
      d.t3.jzt = l->jt + 2 * jn;
      d.t3.ns = 1;
      n = (int64_t)d.t3.ntx * d.t3.nty * l->nsys;
      cost = 2.f + 0.1f * (float)l->L * (float)(d.t3.tx * d.t3.ty) / 64.f;
    } else if (in.form == FORM_2D_WHOLE || in.form == FORM_2D_BANDS) {
      const int rows = kTile2dItems / sa::tile2d_groups(l->L);  // rows of a tile
      const bool whole = in.form == FORM_2D_WHOLE;
      d.m = kSweeps2d;
      d.th = whole ? l->L : std::min(16, rows - 4 * d.m);
      d.bands = whole ? 1 : (l->L + d.th - 1) / d.th;
      for (int64_t e = 0; e < (int64_t)d.bands * l->nsys; ++e) tiles2.push_back(make_int2((int)q, (int)e));
    } else {
      d.form = FORM_HALF;
    }
    if (two_arrays(d.form)) b->desc_m[q] = d.m;
    if (d.form == FORM_2D_WHOLE || d.form == FORM_2D_BANDS) {
      // entries made above
    } else if (d.form == FORM_HALF) {
      for (int64_t off = 0; off < in.work; off += bs) halves.push_back(make_int2((int)q, (int)off));
    } else {
      for (int64_t k = 0; k < n; ++k) tiles.push_back({make_int2((int)q, (int)k), cost});
      total += n * cost;
    }
    if (halves.size() > INT32_MAX / 2 || tiles.size() + tiles2.size() > INT32_MAX / 2) return sa_fail(SA_ERR_ARG, "batch too large");
  }
  // earlier launches may still read the old arrays and the staging buffer
  SA_HIP_TRY(hipStreamSynchronize(b->stream));
  constexpr int nctrl = 2 + 16 + 2;
  const size_t ntile = tiles.size() + tiles2.size();
  bool m1 = false, m2 = false, m3 = false, m4 = false;
  int rc = b->d_desc.ensure(std::max<size_t>(ids.size(), 1), m1);
  if (!rc) rc = b->d_bmap.ensure(std::max<size_t>(halves.size(), 1), m2);
  if (!rc) rc = b->d_ctrl.ensure(nctrl, m3);
  if (!rc) rc = b->d_tmap.ensure(std::max<size_t>(ntile, 1), m4);
  if (rc) return rc;
  if (m1 || m2 || m3 || m4 || b->graph_bs != bs) drop_graphs(b);
  b->graph_bs = bs;
  const size_t o_desc = (sizeof(int) * nctrl + 15) & ~(size_t)15, o_half = o_desc + sizeof(inst_desc) * ids.size();
  const size_t o_tile = o_half + sizeof(int2) * halves.size();
  if (!b->h_stage.ensure(o_tile + sizeof(int2) * ntile + 64)) return sa_fail(SA_ERR_NOMEM, "pinned staging");
  char *st = (char *)b->h_stage.p;
  int *ctrl = (int *)st;
  std::memset(ctrl, 0, sizeof(int) * nctrl);
  ctrl[0] = (int)halves.size();
  ctrl[1] = (int)ids.size();
  // the entries in order, an eighth of the cost to each XCD
  double sum = 0;
  int2 *tmap = (int2 *)(st + o_tile);
  for (size_t e = 0; e < tiles.size(); ++e) {
    const int x = std::min(7, (int)(8 * sum / total));
    if (ctrl[3 + 2 * x]++ == 0) ctrl[2 + 2 * x] = (int)e;
    tmap[e] = tiles[e].e;
    sum += tiles[e].cost;
  }
  ctrl[18] = (int)tiles.size();
  ctrl[19] = (int)tiles2.size();
  std::memcpy(tmap + tiles.size(), tiles2.data(), sizeof(int2) * tiles2.size());
  std::memcpy(st + o_desc, descs.data(), sizeof(inst_desc) * ids.size());
  std::memcpy(st + o_half, halves.data(), sizeof(int2) * halves.size());
  SA_HIP_TRY(hipMemcpyAsync(b->d_ctrl.p, ctrl, sizeof(int) * nctrl, hipMemcpyHostToDevice, b->stream));
  if (!ids.empty())
    SA_HIP_TRY(hipMemcpyAsync(b->d_desc.p, st + o_desc, sizeof(inst_desc) * ids.size(), hipMemcpyHostToDevice, b->stream));
  if (!halves.empty())
    SA_HIP_TRY(hipMemcpyAsync(b->d_bmap.p, st + o_half, sizeof(int2) * halves.size(), hipMemcpyHostToDevice, b->stream));
  if (ntile)
    SA_HIP_TRY(hipMemcpyAsync(b->d_tmap.p, tmap, sizeof(int2) * ntile, hipMemcpyHostToDevice, b->stream));
  b->ndesc = (int)ids.size();
  b->desc_id = ids;
  b->nblocks = (int)halves.size();
  b->ntiles = (int)tiles.size();
  b->ntiles2 = (int)tiles2.size();
  b->bmap_bs = bs;
  b->dirty = false;
  return SA_OK;
}

// One sweep = a launch of the 3D tiles and two half-sweep launches, of whichever there are,
// with a launch of the 2D tiles every kSweeps2d sweeps; the chunk ends with the advance.
int enqueue_sweeps(sa_batch *b, int k) {
  const int grid = grid_for(b, b->bmap_bs);
  const int tgrid = std::max(8, b->cus / 4 * 8);  // two blocks per CU, a multiple of the 8 XCDs
  for (int s = 0; s < k; ++s) {
    if (b->ntiles)
      hipLaunchKernelGGL(k_batch_tile3d, dim3(tgrid), dim3(kTileThreads), kTileLds, b->stream, b->d_desc.p, b->d_tmap.p,
                         b->d_ctrl.p, k, s);
    if (b->ntiles2 && s % kSweeps2d == 0)
      hipLaunchKernelGGL(k_batch_tile2d, dim3(2 * b->cus), dim3(kTile2dThreads), kTile2dItems * 32, b->stream, b->d_desc.p,
                         b->d_tmap.p, b->d_ctrl.p, k, s / kSweeps2d);
    for (int color = 0; color < 2 && b->nblocks; ++color)
      hipLaunchKernelGGL(k_batch_half, dim3(grid), dim3(b->bmap_bs), 0, b->stream, b->d_desc.p, b->d_bmap.p,
                         b->d_ctrl.p, color, s);
  }
  hipLaunchKernelGGL(k_batch_advance, dim3(1), dim3(256), 0, b->stream, b->d_desc.p, b->d_ctrl.p, k);
  return SA_OK;
}

// the graph of k sweeps over the current device arrays (captured on first use)
int graph_for(sa_batch *b, int k, hipGraphExec_t &out) {
  const std::pair<int, int> key(k, (b->ntiles ? 1 : 0) + (b->nblocks ? 2 : 0) + (b->ntiles2 ? 4 : 0));
  auto it = b->graphs.find(key);
  if (it != b->graphs.end()) {
    out = it->second;
    return SA_OK;
  }
  hipGraph_t g = nullptr;
  // more than 64 KB of dynamic LDS has to be asked for
  static sa::per_device_once once;
  SA_HIP_TRY((hipError_t)once(b->device, [] {
    return hipFuncSetAttribute((const void *)k_batch_tile3d, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTileLds);
  }));
  SA_HIP_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  const int erc = enqueue_sweeps(b, k);
  const hipError_t ee = hipStreamEndCapture(b->stream, &g);
  if (erc) {
    if (g) (void)hipGraphDestroy(g);
    return erc;
  }
  SA_HIP_TRY(ee);
  hipGraphExec_t e = nullptr;
  const hipError_t rc = hipGraphInstantiate(&e, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (rc != hipSuccess) return sa_fail(SA_ERR_HIP, "hipGraphInstantiate: %s", hipGetErrorString(rc));
  b->graphs[key] = e;
  out = e;
  return SA_OK;
}

int64_t bonds(const sa_ladder *l) {
  return (l->kind == SA_KIND_3D ? 3 : 2) * l->N - (l->kind == SA_KIND_2P ? l->L : 0);
}

// measure systems sys[j] of instances ids[j]: E/M[j*64 + lane]
int measure_many(sa_batch *b, const std::vector<int> &ids, const std::vector<int> &sys, std::vector<int32_t> &E,
                 std::vector<int32_t> &M) {
  const int n = (int)ids.size();
  E.assign((size_t)n * 64, 0);
  M.assign((size_t)n * 64, 0);
  if (n == 0) return SA_OK;
  std::vector<meas_item> items;
  for (int j = 0; j < n; ++j) {
    const sa_ladder *l = b->inst[ids[j]].lad;
    for (int64_t beg = 0; beg < l->N; beg += kMeasSites) {
      meas_item it;
      std::memset(&it, 0, sizeof it);
      it.s = l->s + (int64_t)sys[j] * l->N;
      it.jx = l->jx;
      it.jy = l->jy;
      it.jz = l->jz;
      it.N = l->N;
      it.begin = beg;
      it.kind = l->kind;
      it.L = l->L;
      it.slot = j;
      items.push_back(it);
    }
  }
  SA_HIP_TRY(hipStreamSynchronize(b->stream));  // the staging buffer may still be read
  bool moved = false;
  int rc = b->d_meas.ensure(items.size(), moved);
  if (!rc) rc = b->d_cnt.ensure((size_t)n * 128, moved);
  if (rc) return rc;
  if (!b->h_stage.ensure(sizeof(meas_item) * items.size())) return sa_fail(SA_ERR_NOMEM, "pinned staging");
  if (!b->h_cnt.ensure(sizeof(int) * n * 128)) return sa_fail(SA_ERR_NOMEM, "pinned staging");
  std::memcpy(b->h_stage.p, items.data(), sizeof(meas_item) * items.size());
  SA_HIP_TRY(hipMemcpyAsync(b->d_meas.p, b->h_stage.p, sizeof(meas_item) * items.size(), hipMemcpyHostToDevice,
                            b->stream));
  hipLaunchKernelGGL(sa::k_fill_zero, dim3((n * 128 + 255) / 256), dim3(256), 0, b->stream, b->d_cnt.p, n * 128);
  hipLaunchKernelGGL(k_batch_measure, dim3((unsigned)items.size()), dim3(256), 0, b->stream, b->d_meas.p,
                     b->d_cnt.p);
  SA_HIP_TRY(hipGetLastError());
  SA_HIP_TRY(hipMemcpyAsync(b->h_cnt.p, b->d_cnt.p, sizeof(int) * n * 128, hipMemcpyDeviceToHost, b->stream));
  SA_HIP_TRY(hipStreamSynchronize(b->stream));
  const int *cnt = (const int *)b->h_cnt.p;
  for (int j = 0; j < n; ++j) {
    const sa_ladder *l = b->inst[ids[j]].lad;
    const int64_t nb = bonds(l);
    for (int k = 0; k < 64; ++k) {
      E[j * 64 + k] = (int32_t)(2 * (int64_t)cnt[j * 128 + k] - nb);
      M[j * 64 + k] = (int32_t)(2 * (int64_t)cnt[j * 128 + 64 + k] - l->N);
    }
  }
  return SA_OK;
}

// exchange step of every listed parallel-tempering instance (parallel_tempering::
// step after its sweeps, src/parallel_tempering.hpp:81-115)
int pt_exchange(sa_batch *b, const std::vector<int> &due) {
  if (due.empty()) return SA_OK;
  std::vector<int> ids, sys;
  for (int id : due) {
    batch_inst &in = b->inst[id];
    in.pt.pend_i = sa::uniform_int(in.pt.gen, 0, in.pt.uni_b);
    in.pt.pend_u = sa::canonical32(in.pt.gen);
    for (int s : {0, in.pt.pend_i, in.pt.pend_i + 1}) {
      ids.push_back(id);
      sys.push_back(s);
    }
  }
  std::vector<int32_t> E, M;
  int rc = measure_many(b, ids, sys, E, M);
  if (rc) return rc;
  std::vector<swap_item> items;
  for (size_t q = 0; q < due.size(); ++q) {
    batch_inst &in = b->inst[due[q]];
    pt_state &p = in.pt;
    float e[3][64];
    for (int r = 0; r < 3; ++r)
      for (int k = 0; k < 64; ++k)
        e[r][k] = (float)((double)E[(q * 3 + r) * 64 + k] + p.h * (double)M[(q * 3 + r) * 64 + k]);
    if (p.E_min.empty()) p.E_min.assign(e[0], e[0] + 64);
    for (int k = 0; k < 64; ++k) p.E_min[k] = std::max(e[0][k], p.E_min[k]);
    const int i = p.pend_i;
    const double dB = 1. / p.T[i] - 1. / p.T[i + 1];
    int acc = 0;
    const uint64_t mask = sa::exchange_word(e[1], e[2], dB, p.pend_u, 64, acc);
    p.acc_sum[i] += acc / 64.0;
    p.acc_n[i] += 1;
    p.pairs.push_back(i);
    p.us.push_back(p.pend_u);
    p.masks.push_back(mask);
    if (!mask) continue;
    const sa_ladder *l = in.lad;
    for (int64_t beg = 0; beg < l->N; beg += kSwapWords) {
      swap_item it;
      it.a = l->s + (int64_t)i * l->N;
      it.b = l->s + (int64_t)(i + 1) * l->N;
      it.mask = mask;
      it.begin = beg;
      it.end = std::min<int64_t>(l->N, beg + kSwapWords);
      items.push_back(it);
    }
  }
  if (items.empty()) return SA_OK;
  bool moved = false;
  rc = b->d_swap.ensure(items.size(), moved);
  if (rc) return rc;
  if (!b->h_stage.ensure(sizeof(swap_item) * items.size())) return sa_fail(SA_ERR_NOMEM, "pinned staging");
  std::memcpy(b->h_stage.p, items.data(), sizeof(swap_item) * items.size());
  SA_HIP_TRY(hipMemcpyAsync(b->d_swap.p, b->h_stage.p, sizeof(swap_item) * items.size(), hipMemcpyHostToDevice,
                            b->stream));
  hipLaunchKernelGGL(k_batch_swap, dim3((unsigned)items.size()), dim3(256), 0, b->stream, b->d_swap.p);
  SA_HIP_TRY(hipGetLastError());
  // every later writer of the staging buffer synchronises the stream first
  return SA_OK;
}

// host mirror of the device sweep indices after k more sweeps; collects the
// parallel-tempering instances whose exchange is due
void advance_host(sa_batch *b, int k, std::vector<int> &due) {
  for (size_t q = 0; q < b->desc_id.size(); ++q) {
    const int id = b->desc_id[q];
    batch_inst &in = b->inst[id];
    if (!in.live) continue;
    const int before = in.t;
    in.t = std::min(in.nsweeps, in.t + k);
    in.lad->t = (uint64_t)in.t;
    const int m = b->desc_m[q], done = in.t - before;
    if (m && ((done + m - 1) / m & 1)) std::swap(in.lad->s, in.lad->s_alt);  // each visit wrote the other array
    if (in.t >= in.nsweeps && before < in.nsweeps) b->dirty = true;
    if (in.pt.every && in.t > before && in.t % in.pt.every == 0) due.push_back(id);
  }
}

int sync_batch(sa_batch *b) {
  SA_HIP_TRY(hipStreamSynchronize(b->stream));
  return SA_OK;
}

// frees what only the tile forms use (the ladder's stream must be idle)
void drop_extras(sa_ladder *l) {
  if (l->s_alt) (void)hipFree(l->s_alt);
  if (l->jt) (void)hipFree(l->jt);
  l->s_alt = nullptr;
  l->jt = nullptr;
  l->jt_current = false;
}

// Everything an instance needs on the device, done without touching the batch (so
// it may run on any thread, while chunks execute): its ladder seeded like main,
// tables uploaded on the ladder's own stream.
int prepare_instance(int kind, int L, int nsys, uint64_t seed, int nsweeps, const double *T, int per_sweep, double h,
                     const pt_state *pt, bool tiles, batch_inst &in) {
  sa_ladder *l = nullptr;
  int rc = sa_ladder_create(kind, L, nsys, &l);
  if (rc) return rc;
  sa_ladder_set_rng(l, SA_RNG_COUNTER);
  // set_seed, init_J, set_seed, init_rand (src/main_gpu.cu:262-276)
  sa_ladder_seed(l, seed);
  rc = sa_ladder_init_couplings(l);
  if (!rc) rc = sa_ladder_seed(l, seed);
  if (!rc) rc = sa_ladder_init_spins(l);
  const int ntab = per_sweep ? std::max(1, nsweeps) * nsys : nsys;
  std::vector<sa::sys_table> tabs(ntab);
  std::vector<char> fasts(ntab);
  bool fast = true;
  for (int q = 0; q < ntab && !rc; ++q) {
    bool f = false;
    sa_detail::make_table(kind, T[per_sweep && nsweeps == 0 ? q % nsys : q], h, tabs[q], f, nullptr);
    fasts[q] = f;
    fast = fast && f;
  }
  // what the tiles need beside the instance's own arrays; without it, half-sweeps
  int form = !rc && fast && tiles ? tile_form(kind, L) : FORM_HALF;
  if (two_arrays(form) && hipMalloc(&l->s_alt, (size_t)nsys * l->N * 8) != hipSuccess) {
    l->s_alt = nullptr;
    (void)hipGetLastError();
    form = FORM_HALF;
  }
  if (form && kind == SA_KIND_3D && !sa_detail::tile3d_couplings(l)) {
    drop_extras(l);
    form = FORM_HALF;
  }
  in = batch_inst();
  in.lad = l;
  in.nsweeps = nsweeps;
  in.per_sweep = per_sweep ? 1 : 0;
  in.fast = fast;
  in.form = form;
  in.work = (int64_t)half_items(kind, L) * nsys;
  if (!rc && hipMalloc(&in.tabs, sizeof(sa::sys_table) * ntab) != hipSuccess) rc = sa_fail(SA_ERR_NOMEM, "tables");
  // on the ladder's stream (waited for below): admission may run while a chunk is
  // on the batch stream, and a null-stream copy would wait for it
  if (!rc && hipMemcpyAsync(in.tabs, tabs.data(), sizeof(sa::sys_table) * ntab, hipMemcpyHostToDevice,
                            l->stream) != hipSuccess)
    rc = sa_fail(SA_ERR_HIP, "table upload");
  // fixed temperatures also become the ladder's own tables, for plain sweeps later
  if (!rc && !per_sweep) rc = sa_detail::ladder_tables(l, std::move(tabs), std::move(fasts));
  if (!rc) rc = sa_ladder_sync(l);
  if (rc) {
    if (in.tabs) (void)hipFree(in.tabs);
    sa_ladder_destroy(l);
    in = batch_inst();
    return rc;
  }
  in.bytes = sa_detail::batch_instance_bytes(kind, L, nsys, nsweeps, per_sweep) + form_bytes(kind, L, nsys, form);
  if (pt) in.pt = *pt;
  return SA_OK;
}

void attach_instance(sa_batch *b, batch_inst &&in, int *id) {
  in.live = true;
  b->bytes_live += in.bytes;
  b->inst.push_back(std::move(in));
  *id = (int)b->inst.size() - 1;
  b->dirty = true;
}

int add_instance(sa_batch *b, int kind, int L, int nsys, uint64_t seed, int nsweeps, const double *T, int per_sweep,
                 double h, pt_state *pt, int *id) {
  batch_inst in;
  int rc = prepare_instance(kind, L, nsys, seed, nsweeps, T, per_sweep, h, pt, true, in);
  if (rc == SA_ERR_NOMEM) {
    // the instances' tile arrays give way to a new instance: all go back to half-sweeps, unless
    // even that is too little
    int64_t extras = 0;
    for (const batch_inst &x : b->inst)
      if (x.live) extras += form_bytes(x.lad->kind, x.lad->L, x.lad->nsys, x.form);
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) == hipSuccess &&
        (int64_t)free_b + extras < sa_detail::batch_instance_bytes(kind, L, nsys, nsweeps, per_sweep))
      return rc;
    const int src = sync_batch(b);
    if (src) return src;
    for (batch_inst &x : b->inst)
      if (x.live && x.form) {
        const int64_t own = x.bytes - form_bytes(x.lad->kind, x.lad->L, x.lad->nsys, x.form);
        const int lrc = sa_ladder_sync(x.lad);
        if (lrc) return lrc;
        drop_extras(x.lad);
        x.form = FORM_HALF;
        b->bytes_live += own - x.bytes;
        x.bytes = own;
        b->dirty = true;
      }
    rc = prepare_instance(kind, L, nsys, seed, nsweeps, T, per_sweep, h, pt, false, in);
  }
  if (rc) return rc;
  attach_instance(b, std::move(in), id);
  return SA_OK;
}

// parallel-tempering state as parallel_tempering's constructor sets it up
pt_state make_pt(int nT, const double *T, double h, int every) {
  pt_state p;
  p.every = every;
  p.T.assign(T, T + nT);
  std::sort(p.T.begin(), p.T.end());  // parallel_tempering sorts its temperatures
  p.h = h;
  p.gen.seed(123);
  p.uni_b = nT - 2;
  p.acc_sum.assign(nT - 1, 0.0);
  p.acc_n.assign(nT - 1, 0);
  return p;
}

}  // namespace

struct sa_detail::prepared_instance {
  batch_inst in;
};

namespace sa_detail {
int batch_geometry(int kind, int L, int nsys) {
  if (kind < SA_KIND_2P || kind > SA_KIND_3D) return sa_fail(SA_ERR_ARG, "unknown kind %d", kind);
  if (nsys < 1) return sa_fail(SA_ERR_ARG, "nsys must be >= 1");
  if (L < 3) return sa_fail(SA_ERR_UNSUPPORTED, "device path needs L >= 3 (got %d)", L);
  if ((kind == SA_KIND_3D && L > 1024) || (kind != SA_KIND_3D && L > 32768))
    return sa_fail(SA_ERR_ARG, "L=%d too large", L);
  // k_batch_half and the block map carry an instance's work item in an int
  if ((int64_t)half_items(kind, L) * nsys >= ((int64_t)1 << 31))
    return sa_fail(SA_ERR_UNSUPPORTED, "instance too large for the batch: %lld work items per half-sweep (limit 2^31)",
                   (long long)half_items(kind, L) * nsys);
  return SA_OK;
}

int batch_prepare(int kind, int L, int nsys, uint64_t seed, int nsweeps, const double *T, int per_sweep, double h,
                  int pt_every, bool tiles, prepared_instance **out) {
  *out = nullptr;
  int rc = batch_geometry(kind, L, nsys);
  if (rc) return rc;
  std::unique_ptr<prepared_instance> p(new prepared_instance());
  if (pt_every > 0) {
    if (nsys < 2 || nsweeps % pt_every) return sa_fail(SA_ERR_ARG, "bad parallel-tempering instance");
    pt_state pt = make_pt(nsys, T, h, pt_every);
    rc = prepare_instance(kind, L, nsys, seed, nsweeps, pt.T.data(), 0, h, &pt, tiles, p->in);
  } else {
    rc = prepare_instance(kind, L, nsys, seed, nsweeps, T, per_sweep, h, nullptr, tiles, p->in);
  }
  if (rc) return rc;
  *out = p.release();
  return SA_OK;
}

int batch_attach(sa_batch *b, prepared_instance *p, int *id) {
  attach_instance(b, std::move(p->in), id);
  delete p;
  return SA_OK;
}

void batch_discard(prepared_instance *p) {
  if (!p) return;
  if (p->in.tabs) (void)hipFree(p->in.tabs);
  sa_ladder_destroy(p->in.lad);
  delete p;
}

int64_t batch_instance_bytes(int kind, int L, int nsys, int nsweeps, int per_sweep) {
  const int ntab = per_sweep ? std::max(1, nsweeps) * nsys : nsys;
  return ladder_bytes(kind, L, nsys) + (int64_t)sizeof(sa::sys_table) * ntab;
}

int64_t batch_tile_bytes(int kind, int L, int nsys) { return form_bytes(kind, L, nsys, tile_form(kind, L)); }

int batch_launch_chunk(sa_batch *b, int max_sweeps, int *k_out) {
  *k_out = 0;
  // fixed by the caller, tuned, or the next trial
  int trial = -1;
  if ((!b->block || !b->chunk) && !(b->tuned_block && b->tuned_chunk)) {
    trial = (int)b->trials.size();
    if (trial >= kNumCands) {
      int best = 0;
      for (int q = 1; q < kNumCands; ++q)
        if (b->trials[q].second < b->trials[best].second) best = q;
      b->tuned_block = kCands[best].block;
      b->tuned_chunk = kCands[best].chunk;
      trial = -1;
    }
  }
  const int bs = b->block ? b->block : (trial >= 0 ? kCands[trial].block : b->tuned_block);
  const int kfull = b->chunk ? b->chunk : (trial >= 0 ? kCands[trial].chunk : b->tuned_chunk);
  if (b->dirty || b->bmap_bs != bs) {
    const int rc = rebuild(b, bs);
    if (rc) return rc;
  }
  if (b->ndesc == 0 || max_sweeps <= 0) return SA_OK;
  // the chunk ends at the next exchange point of any parallel-tempering instance
  int64_t k = std::min(kfull, max_sweeps);
  int remaining = 0;
  for (int id : b->desc_id) {
    const batch_inst &in = b->inst[id];
    remaining = std::max(remaining, in.nsweeps - in.t);
    if (in.pt.every) k = std::min<int64_t>(k, in.pt.every - in.t % in.pt.every);
  }
  k = std::min<int64_t>(k, remaining);
  if (k <= 0) return SA_OK;
  hipGraphExec_t g = nullptr;
  int rc = graph_for(b, (int)k, g);
  if (rc) return rc;
  if (trial >= 0) SA_HIP_TRY(hipEventRecord(b->ev0, b->stream));
  SA_HIP_TRY(hipGraphLaunch(g, b->stream));
  if (trial >= 0) {
    SA_HIP_TRY(hipEventRecord(b->ev1, b->stream));
    SA_HIP_TRY(hipEventSynchronize(b->ev1));
    float ms = 0;
    SA_HIP_TRY(hipEventElapsedTime(&ms, b->ev0, b->ev1));
    // time per work item, so trials on different schedules compare
    double work = 0;
    for (int id : b->desc_id)
      work += (double)b->inst[id].work * std::min<int64_t>(k, b->inst[id].nsweeps - b->inst[id].t);
    b->trials.push_back({trial, (float)(ms / std::max(work, 1.0))});
  }
  *k_out = (int)k;
  return SA_OK;
}

int batch_finish_chunk(sa_batch *b, int k) {
  std::vector<int> due;
  advance_host(b, k, due);
  return pt_exchange(b, due);
}

int batch_wait(sa_batch *b) { return sync_batch(b); }

sa_ladder *batch_instance_ladder(sa_batch *b, int id) {
  return (id >= 0 && id < (int)b->inst.size() && b->inst[id].live) ? b->inst[id].lad : nullptr;
}

bool batch_done(const sa_batch *b, int id) {
  return id >= 0 && id < (int)b->inst.size() && b->inst[id].live && b->inst[id].t >= b->inst[id].nsweeps;
}
}  // namespace sa_detail

extern "C" {

int sa_batch_create(sa_batch **out) {
  if (!out) return sa_fail(SA_ERR_ARG, "null output handle");
  sa_batch *b = new sa_batch();
  hipDeviceProp_t prop;
  if (hipGetDevice(&b->device) == hipSuccess && hipGetDeviceProperties(&prop, b->device) == hipSuccess &&
      prop.multiProcessorCount > 0)
    b->cus = prop.multiProcessorCount;
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess || hipEventCreate(&b->ev0) != hipSuccess ||
      hipEventCreate(&b->ev1) != hipSuccess) {
    delete b;
    return sa_fail(SA_ERR_HIP, "stream/event creation failed");
  }
  *out = b;
  return SA_OK;
}

int sa_batch_destroy(sa_batch *b) {
  if (!b) return SA_OK;
  (void)hipStreamSynchronize(b->stream);
  drop_graphs(b);
  for (auto &in : b->inst)
    if (in.live) {
      if (in.tabs) (void)hipFree(in.tabs);
      sa_ladder_destroy(in.lad);
    }
  if (b->ev0) (void)hipEventDestroy(b->ev0);
  if (b->ev1) (void)hipEventDestroy(b->ev1);
  hipStream_t s = b->stream;
  delete b;  // device arrays and staging buffers free themselves
  (void)hipStreamDestroy(s);
  return SA_OK;
}

int sa_batch_add(sa_batch *b, int kind, int L, int nsys, uint64_t seed, int nsweeps, const double *T, int per_sweep,
                 double h, int *id) {
  const int rc = sa_detail::batch_geometry(kind, L, nsys);  // before anything touches the device
  if (rc) return rc;
  if (!b || !T || !id || nsweeps < 0) return sa_fail(SA_ERR_ARG, "bad argument");
  return add_instance(b, kind, L, nsys, seed, nsweeps, T, per_sweep, h, nullptr, id);
}

int sa_batch_add_pt(sa_batch *b, int kind, int L, int nT, const double *T, double h, uint64_t seed, int every,
                    int nsteps, int *id) {
  const int rc = sa_detail::batch_geometry(kind, L, nT);  // before anything touches the device
  if (rc) return rc;
  if (!b || !T || !id || nT < 2 || every < 1 || nsteps < 0) return sa_fail(SA_ERR_ARG, "bad argument");
  if ((int64_t)every * nsteps > INT32_MAX / 2) return sa_fail(SA_ERR_ARG, "too many sweeps");
  pt_state p = make_pt(nT, T, h, every);
  return add_instance(b, kind, L, nT, seed, every * nsteps, p.T.data(), 0, h, &p, id);
}

int sa_batch_run(sa_batch *b, int sweeps) {
  if (!b) return sa_fail(SA_ERR_ARG, "null batch");
  // Between two runs a ladder that was handed out may have been swept (on its own stream, and
  // into its other spin array), given other couplings or seeded: wait for it and schedule anew.
  for (const batch_inst &in : b->inst)
    if (in.live && in.lent) {
      SA_HIP_TRY(hipStreamSynchronize(in.lad->stream));
      b->dirty = true;
    }
  int64_t left = sweeps > 0 ? sweeps : INT64_MAX;
  while (left > 0) {
    int k = 0;
    int rc = sa_detail::batch_launch_chunk(b, (int)std::min<int64_t>(left, INT32_MAX), &k);
    if (rc) return rc;
    if (k == 0) break;
    rc = sa_detail::batch_finish_chunk(b, k);
    if (rc) return rc;
    left -= k;
  }
  int rc = sync_batch(b);
  if (rc) return rc;
  int unfinished = 0;
  for (auto &in : b->inst)
    if (in.live && in.t < in.nsweeps) ++unfinished;
  return unfinished;
}

int sa_batch_sweeps_done(sa_batch *b, int id, int *t) {
  int rc = check_id(b, id);
  if (rc) return rc;
  if (!t) return sa_fail(SA_ERR_ARG, "null argument");
  *t = b->inst[id].t;
  return SA_OK;
}

int sa_batch_get_spins(sa_batch *b, int id, int sys, uint64_t *s) {
  int rc = check_id(b, id);
  if (rc) return rc;
  rc = sync_batch(b);
  if (rc) return rc;
  return sa_ladder_get_spins(b->inst[id].lad, sys, s);
}

int sa_batch_measure(sa_batch *b, int id, int32_t *E, int32_t *M) {
  int rc = check_id(b, id);
  if (rc) return rc;
  rc = sync_batch(b);
  if (rc) return rc;
  return sa_ladder_measure(b->inst[id].lad, E, M);
}

int sa_batch_pt_result(sa_batch *b, int id, int64_t capacity, int32_t *pairs, double *us, uint64_t *masks,
                       float *E_min, double *acceptance) {
  int rc = check_id(b, id);
  if (rc) return rc;
  const pt_state &p = b->inst[id].pt;
  if (!p.every) return sa_fail(SA_ERR_STATE, "instance %d is not a parallel-tempering instance", id);
  const int64_t n = std::min<int64_t>(capacity, (int64_t)p.pairs.size());
  for (int64_t k = 0; k < n; ++k) {
    if (pairs) pairs[k] = p.pairs[k];
    if (us) us[k] = p.us[k];
    if (masks) masks[k] = p.masks[k];
  }
  if (E_min)
    for (int k = 0; k < 64; ++k) E_min[k] = p.E_min.empty() ? 0.f : p.E_min[k];
  if (acceptance)
    for (size_t i = 0; i < p.acc_sum.size(); ++i) acceptance[i] = p.acc_n[i] ? p.acc_sum[i] / p.acc_n[i] : 0.0;
  return (int)std::min<int64_t>((int64_t)p.pairs.size(), INT32_MAX);
}

sa_ladder *sa_batch_ladder(sa_batch *b, int id) {
  if (check_id(b, id)) return nullptr;
  if (sync_batch(b)) return nullptr;
  b->inst[id].lent = true;
  return b->inst[id].lad;
}

int sa_batch_remove(sa_batch *b, int id) {
  int rc = check_id(b, id);
  if (rc) return rc;
  rc = sync_batch(b);
  if (rc) return rc;
  batch_inst &in = b->inst[id];
  if (in.tabs) (void)hipFree(in.tabs);
  sa_ladder_destroy(in.lad);
  b->bytes_live -= in.bytes;
  in = batch_inst();
  b->dirty = true;
  return SA_OK;
}

int64_t sa_batch_bytes(const sa_batch *b) { return b ? b->bytes_live : 0; }

void *sa_batch_stream(sa_batch *b) { return b ? (void *)b->stream : nullptr; }

int sa_batch_set_tuning(sa_batch *b, int key, int value) {
  if (!b) return sa_fail(SA_ERR_ARG, "null batch");
  if (key == SA_TUNE_BATCH_BLOCK) {
    if (value != 0 && value != 64 && value != 128 && value != 256)
      return sa_fail(SA_ERR_ARG, "batch block must be 0 (auto), 64, 128 or 256");
    b->block = value;
  } else if (key == SA_TUNE_BATCH_CHUNK) {
    if (value < 0 || value > 4096) return sa_fail(SA_ERR_ARG, "batch chunk must be 0 (auto) .. 4096");
    b->chunk = value;
  } else if (key == SA_TUNE_BATCH_FUSED) {
    if (value < 0 || value > 2) return sa_fail(SA_ERR_ARG, "batch fused must be 0 (auto), 1 (off) or 2 (on)");
    if (value == 2) return sa_fail(SA_ERR_ARG, "the fused batch sweep is switched off in this build");
  } else {
    return sa_fail(SA_ERR_ARG, "unknown batch tuning key %d", key);
  }
  b->dirty = true;
  return SA_OK;
}

int sa_batch_get_tuning(sa_batch *b, int key, int *value) {
  if (!b || !value) return sa_fail(SA_ERR_ARG, "null argument");
  if (key == SA_TUNE_BATCH_BLOCK) *value = b->block ? b->block : b->tuned_block;
  else if (key == SA_TUNE_BATCH_CHUNK) *value = b->chunk ? b->chunk : b->tuned_chunk;
  else if (key == SA_TUNE_BATCH_FUSED) *value = 1;
  else return sa_fail(SA_ERR_ARG, "unknown batch tuning key %d", key);
  return SA_OK;
}

}  // extern "C"
