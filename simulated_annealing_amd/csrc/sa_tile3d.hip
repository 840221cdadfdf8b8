// sa_tile3d.hip -- choice and launch of the 3D tile sweep (sa_tile3d.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "sa_internal.hpp"
#include "sa_per_device.hpp"
#include "sa_tile3d.hpp"

namespace {

constexpr size_t kMaxLds = 160 * 1024;

struct tile_cfg {
  bool whole;
  int S, threads, ns;
  size_t lds;
  sa::tile3d_args a;  // geometry only
};

// The tile of the next launch: the one with the least modelled time per sweep, in us.
// Fitted to 60 measured shapes (3D L 8..128, 1..32 systems), within 25%: a launch with its
// load and store, a wave's worth of columns, and the tiles' reads and writes at 8 TB/s;
// four-plane segments need half the waves but take about twice as long each.  A tile's work grows with
// its waves, its overhead with its halo: one L=64 system takes 4 x 4 columns (256 tiles, 7.2
// us per sweep; 8 x 8: 11.0), 16 systems of L=32 16 x 4 (7.4; 4 x 4: 10.0, 16 x 8: 8.6).
tile_cfg pick(const sa_ladder *l, int64_t left, double &cost) {
  tile_cfg best{};
  cost = 1e30;
  const int L = l->L;
  if (l->kind != SA_KIND_3D || L > 256) return best;
  const bool odd = L & 1;
  const bool general = std::any_of(l->fast.begin(), l->fast.end(), [](char f) { return !f; });
  auto consider = [&](bool whole, int tx, int ty, int S) {
    tile_cfg c{};
    c.whole = whole;
    c.S = S;
    const int W = whole ? L : tx + 4, H = whole ? L : ty + 4, row = odd ? W : W / 2;
    if (row * H > 1024) return;
    // first for a full block, to learn the waves the columns make
    if (!sa::tile3d_setup(c.a, L, whole, tx, ty, S, 1024)) return;
    c.threads = std::max(std::min(16, c.a.chunks0) * 64, (row * H + 63) / 64 * 64);
    c.lds = sa::tile3d_setup(c.a, L, whole, tx, ty, S, c.threads);
    if (!c.lds || c.lds > kMaxLds) return;
    c.ns = whole ? (int)std::min<int64_t>(left, 64) : 1;
    const int64_t tiles = (int64_t)c.a.ntx * c.a.nty;
    const double per_cu = std::ceil((double)tiles * l->nsys / 256);
    const double wave = S == 2 ? (general ? 0.195 : 0.13) : (general ? 0.29 : 0.25);
    const double words = (double)l->nsys * l->N, amp = (double)(W * H) / (c.a.tx * c.a.ty);
    // odd sides: up to three more stages
    const double stages = odd ? 2.5 : 0;
    const double t = ((S == 2 ? 4.6 : 6.3) + words * 8 * (amp + 1) / 8e6) / c.ns + stages +
                     per_cu * (c.a.chunks0 + c.a.chunks1) * wave;
    if (t < cost) {
      cost = t;
      best = c;
    }
  };
  for (int S : {2, 4}) {
    if (S == 2) consider(true, L, L, S);
    for (int tx : {4, 8, 16, 32})
      for (int ty : {4, 8, 16, 32})
        if (tx <= L && ty <= L) consider(false, tx, ty, S);
  }
  return best;
}

// more than 64 KB of dynamic LDS has to be asked for, once per kernel and device
template <class K>
int allow_lds(sa::per_device_once &once, int device, K kernel) {
  return once(device, [&] {
    return hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
  });
}

// 0 or the error of the LDS request (nothing launched)
template <bool COUNTER, bool FAST, int S>
int launch(const sa::tile3d_args &t, const tile_cfg &c, int device, hipStream_t st) {
  const dim3 grid((unsigned)((t.ntx * t.nty * t.a.nsys + 7) / 8 * 8));
  const size_t lds = c.lds;
  auto go = [&](auto whole, auto one) {
    constexpr auto kernel = sa::k_tile3d<COUNTER, FAST, S, decltype(whole)::value, decltype(one)::value>;
    static sa::per_device_once once;
    if (const int e = allow_lds(once, device, kernel)) return e;
    hipLaunchKernelGGL(kernel, grid, dim3(c.threads), lds, st, t);
    return 0;
  };
  if (t.a.L & 1) {
    auto go_odd = [&](auto whole) {
      constexpr auto kernel = sa::k_tile3d_odd<COUNTER, FAST, S, decltype(whole)::value>;
      static sa::per_device_once once;
      if (const int e = allow_lds(once, device, kernel)) return e;
      hipLaunchKernelGGL(kernel, grid, dim3(c.threads), lds, st, t);
      return 0;
    };
    return c.whole ? go_odd(std::true_type{}) : go_odd(std::false_type{});
  }
  const bool one = c.a.chunks0 * 64 <= c.threads;
  if constexpr (S == 2) {  // the kept couplings fit the registers
    if (one) return c.whole ? go(std::true_type{}, std::true_type{}) : go(std::false_type{}, std::true_type{});
  }
  return c.whole ? go(std::true_type{}, std::false_type{}) : go(std::false_type{}, std::false_type{});
}

// in (rows x cols) to out (cols x rows, `stride` words per row), 32 x 32 words at a time;
// blockIdx.z: the array
__global__ void __launch_bounds__(256) k_transpose(const uint64_t *__restrict__ in, uint64_t *__restrict__ out, int rows,
                                                   int cols, int stride) {
  __shared__ uint64_t tile[32][33];
  const int64_t base = (int64_t)blockIdx.z * rows * cols, obase = (int64_t)blockIdx.z * stride * cols;
  const int c0 = (int)blockIdx.x * 32, r0 = (int)blockIdx.y * 32, i = (int)threadIdx.x & 31, j0 = (int)threadIdx.x >> 5;
  for (int j = j0; j < 32; j += 8)
    if (r0 + j < rows && c0 + i < cols) tile[j][i] = in[base + (int64_t)(r0 + j) * cols + c0 + i];
  __syncthreads();
  for (int j = j0; j < 32; j += 8)
    if (c0 + j < cols && r0 + i < rows) out[obase + (int64_t)(c0 + j) * stride + r0 + i] = tile[i][j];
}

}  // namespace

// the ladder's couplings with z fastest, on its stream; false without memory
bool sa_detail::tile3d_couplings(sa_ladder *l) {
  const int stride = sa::column_stride(l->L);
  if (!l->jt && hipMalloc(&l->jt, (size_t)3 * l->L * l->L * stride * 8) != hipSuccess) {
    l->jt = nullptr;
    (void)hipGetLastError();
    return false;
  }
  if (l->jt_current) return true;
  const int L2 = l->L * l->L;
  hipLaunchKernelGGL(k_transpose, dim3((unsigned)((L2 + 31) / 32), (unsigned)((l->L + 31) / 32), 3), dim3(256), 0,
                     l->stream, l->jx, l->jt, l->L, L2, stride);
  l->jt_current = true;
  return true;
}

int sa_detail::tile3d_sweeps(const sa_ladder *l, int64_t left, bool *second, double *us) {
  double cost = 0;
  const tile_cfg c = pick(l, left, cost);
  *second = c.S > 0 && !c.whole;
  *us = cost;
  return c.S > 0 ? c.ns : 0;
}

int sa_detail::tile3d_launch(sa_ladder *l, const sa::sys_table *tab, int64_t tab_step, bool fast, const uint64_t *words,
                             uint64_t t, int64_t left) {
  double cost = 0;
  const tile_cfg c = pick(l, left, cost);
  sa::tile3d_args a = c.a;
  a.a.s = l->s;
  a.a.jx = l->jx;
  a.a.jy = l->jy;
  a.a.jz = l->jz;
  a.a.tab = tab;
  a.a.words = words;
  a.a.seed = l->seed;
  a.a.sweep = t;
  a.a.N = l->N;
  a.a.L = l->L;
  a.a.nsys = l->nsys;
  a.out = c.whole ? l->s : l->s_alt;
  a.jxt = l->jt;
  const int64_t jn = (int64_t)l->L * l->L * sa::column_stride(l->L);
  a.jyt = l->jt + jn;
  a.jzt = l->jt + 2 * jn;
  a.ns = c.ns;
  a.tab_step = tab_step;
  const bool counter = l->rng_mode == SA_RNG_COUNTER;
#define SA_T3(CO, FA)                                                                                             \
  if (counter == CO && fast == FA)                                                                                \
    e = c.S == 2 ? launch<CO, FA, 2>(a, c, l->device, l->stream) : launch<CO, FA, 4>(a, c, l->device, l->stream);
  const int64_t most = sa::systems_per_launch((uint32_t)(a.ntx * a.nty), c.threads);
  for (int64_t left_sys = l->nsys; left_sys > 0;) {
    int e = 0;
    a.a.nsys = (int)std::min(left_sys, most);
    SA_T3(true, true)
    SA_T3(true, false)
    SA_T3(false, true)
    SA_T3(false, false)
    if (e) return sa_fail(SA_ERR_HIP, "LDS of the 3D tiles: %s", hipGetErrorString((hipError_t)e));
    left_sys -= a.a.nsys;
    a.a.s += a.a.nsys * l->N;
    a.out += a.a.nsys * l->N;
    a.a.tab += a.a.nsys;
  }
#undef SA_T3
  if (!c.whole) std::swap(l->s, l->s_alt);
  return SA_OK;
}
