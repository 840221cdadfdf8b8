// sa_tile2d.hip -- choice and launch of the 2D sweeps held in LDS (sa_tile2d.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sa_internal.hpp"
#include "sa_tile2d.hpp"
#include "sa_tile_place.hpp"

namespace {

constexpr int kMaxSide = 768;
constexpr int kMaxItems = 2048;  // items of a tile (32 B of LDS each): two per thread of 1024

struct tile_cfg {
  bool wrap;
  int th, ns, bands, items;  // ns: sweeps per launch
};

size_t tile_lds(int L, int rows) { return (size_t)rows * 2 * sa::tile2d_half(L) * 8; }

// The tile of the next launch: the one with the least modelled time per sweep, in us.
// A launch costs 3.3 us plus its tiles' reads (spins 8 B, couplings 32 B per word, mostly
// from L2) and writes at 12 TB/s; a half-sweep 0.38 us plus 0.047 us per wave of items on
// a CU (fitted to 24 measured shapes, L 16..512, 1..32 systems, within 20%).  So small
// lattices take one workgroup per system and as many sweeps as asked for, larger ones
// bands of 4..16 rows and 2..5 sweeps.  Against the half-sweep kernels (us per sweep, half-sweep
// kernels / here): 2D L=64 1 system 7.2 / 2.0, 24 systems 9.9 / 2.0; L=128 x16 10.4 / 2.7;
// L=256 x32 25 / 10.5; L=512 x1 13 / 8.7, x32 112 / 55; open x with a field L=256 x8 20.7 / 7.0.
// Up to kMaxSide two sweeps fit a launch; above it one does (L=1024 x32 with a field 444 / 452).
tile_cfg pick(const sa_ladder *l, int64_t left) {
  tile_cfg best{false, 0, 0, 0, 0};
  // asked for a number of systems per thread: the half-sweep kernels, which have that choice
  if (l->kind == SA_KIND_3D || l->L > kMaxSide || l->sys_per_thread > 0) return best;
  if (l->L & 1) {  // odd sides: the whole lattice (up to 89, always the faster) or not at all
    const int items = l->L * sa::tile2d_groups(l->L);
    return items <= kMaxItems ? tile_cfg{true, l->L, (int)std::min<int64_t>(left, 64), 1, items} : best;
  }
  const int L = l->L, G = sa::tile2d_groups(L);
  double cost = 1e30;
  auto consider = [&](bool wrap, int th, int ns) {
    const int rows = wrap ? L : th + 4 * ns, items = rows * G, bands = wrap ? 1 : (L + th - 1) / th;
    if (items > kMaxItems) return;
    const double wgs = (double)l->nsys * bands, waves = ((items + 63) / 64) * std::max(1.0, wgs / 256);
    const double half = 0.38 + 0.047 * waves;
    const double words = (double)l->nsys * bands * rows * L;  // read: spins, couplings (mostly from L2)
    const double c = (3.3 + (40 * words + 8.0 * l->nsys * l->N) / 12e6) / ns + 2 * half;
    if (c < cost) {
      cost = c;
      best = tile_cfg{wrap, wrap ? L : th, ns, bands, items};
    }
  };
  consider(true, L, (int)std::min<int64_t>(left, 64));
  for (int th : {2, 4, 8, 16, 32, 64})
    for (int ns : {1, 2, 3, 4, 5, 8, 10})
      if (ns <= left) consider(false, th, ns);
  return best;
}

template <bool COUNTER, int MODE, int IT>
void launch(const sa::tile2d_args &t, bool wrap, int threads, size_t lds, hipStream_t st) {
  const dim3 grid((unsigned)(t.a.nsys * t.bands));
  if (t.a.L & 1) {
    hipLaunchKernelGGL((sa::k_tile2d_odd<COUNTER, MODE, IT>), grid, dim3(threads), lds, st, t);
  } else if (wrap) {
    hipLaunchKernelGGL((sa::k_tile2d<COUNTER, MODE, IT, true>), grid, dim3(threads), lds, st, t);
  } else {
    hipLaunchKernelGGL((sa::k_tile2d<COUNTER, MODE, IT, false>), grid, dim3(threads), lds, st, t);
  }
}

template <bool COUNTER, int MODE>
void launch_it(const sa::tile2d_args &t, const tile_cfg &c, hipStream_t st) {
  const int threads = std::min(1024, (c.items + 63) / 64 * 64);
  const size_t lds = (t.a.L & 1) ? (size_t)t.a.L * t.a.L * 8 : tile_lds(t.a.L, c.wrap ? t.a.L : c.th + 4 * t.ns);
  if (c.items <= threads) launch<COUNTER, MODE, 1>(t, c.wrap, threads, lds, st);
  else launch<COUNTER, MODE, 2>(t, c.wrap, threads, lds, st);
}

}  // namespace

int sa_detail::tile2d_sweeps(const sa_ladder *l, int64_t left, bool *bands) {
  const tile_cfg c = pick(l, left);
  *bands = c.ns > 0 && !c.wrap;
  return c.ns;
}

void sa_detail::tile2d_launch(sa_ladder *l, const sa::sys_table *tab, int64_t tab_step, bool fast, const uint64_t *words,
                              uint64_t t, int64_t left, int ns) {
  const tile_cfg c = pick(l, left);
  sa::tile2d_args a;
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
  a.out = c.wrap ? l->s : l->s_alt;
  a.ns = ns;
  a.th = c.th;
  a.bands = c.bands;
  a.tab_step = tab_step;
  const bool counter = l->rng_mode == SA_RNG_COUNTER;
  const int mode = l->kind == SA_KIND_2P ? sa::T2_OPEN : fast ? sa::T2_FAST : sa::T2_GENERAL;
#define SA_T2(C, M) \
  if (counter == C && mode == M) launch_it<C, M>(a, c, l->stream)
  const int64_t most = sa::systems_per_launch((uint32_t)c.bands, 1024);  // 4 million lattices held whole
  for (int64_t left_sys = l->nsys; left_sys > 0;) {
    a.a.nsys = (int)std::min(left_sys, most);
    SA_T2(true, sa::T2_FAST);
    SA_T2(true, sa::T2_GENERAL);
    SA_T2(true, sa::T2_OPEN);
    SA_T2(false, sa::T2_FAST);
    SA_T2(false, sa::T2_GENERAL);
    SA_T2(false, sa::T2_OPEN);
    left_sys -= a.a.nsys;
    a.a.s += a.a.nsys * l->N;
    a.out += a.a.nsys * l->N;
    a.a.tab += a.a.nsys;
  }
#undef SA_T2
  if (!c.wrap) std::swap(l->s, l->s_alt);
}
