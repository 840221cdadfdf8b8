// sa_tile2d.hpp -- several 2D sweeps per launch with the lattice held in LDS (even L; odd L
// where it fits whole, further down).
//
// What bounds a 2D lattice of ordinary size is not memory but launches: one half-sweep
// per launch costs 3-4 us of which the update is a fraction.  Here a workgroup keeps a
// tile in LDS through `ns` whole sweeps and touches memory only at the start and the end:
//   WRAP: the whole lattice (at most 2048 items, L up to 88), updated in place; one workgroup per system.
//   bands: TH full rows plus 2*ns halo rows on either side.  Half-sweep h (0 .. 2*ns-1)
//     updates the rows at least h+1 away from the tile's edge, so after ns sweeps the TH
//     rows in the middle are exact and the halo's have been recomputed redundantly (the
//     same words the neighbouring bands compute).  Bands read one spin array and write
//     another, so no workgroup waits for another.
// Every word is the one the two launches of a half-sweep pair produce: a half-sweep reads
// only words of the other colour and the site's own (even L), and a site's random word
// depends on its coordinates and the sweep only.
//
// A thread owns `IT` items; an item is four neighbouring columns of one row, i.e. the pair
// (x, x+2) of either colour -- the pair one Philox block serves -- with its couplings in
// registers for the whole launch.  LDS keeps a row as its even columns followed by its odd
// ones, so a pair, its +-y neighbours and two of its three x neighbours are 128-bit
// accesses to consecutive lanes' consecutive addresses (no bank conflicts).
//
// With the launches gone the update itself is the bound: a wave of items takes about 450
// cycles of its SIMD per half-sweep (one Philox block, two updates), a half-sweep of one
// wave 0.4 us (a chain of the block's ten rounds, LDS and the update).  2D L=64, 24
// systems: 9.9 -> 2.0 us per sweep; tables with a field by counting accepted levels
// instead of two select trees: open-x L=256, 8 systems 20.7 -> 7.0 us.
#pragma once

#include "sa_kernels.hpp"

namespace sa {

struct tile2d_args {
  sweep_args a;       // a.sweep: index of the first sweep; a.words: replay words of that sweep
  uint64_t *out;      // bands: the array written (WRAP: a.s itself)
  int ns;             // sweeps of this launch
  int th;             // rows per band (WRAP: L)
  int bands;          // bands per system (WRAP: 1)
  int64_t tab_step;   // tables per sweep (0: one temperature for all sweeps)
};

// LDS words of one row: two half rows, each padded to an even length (128-bit accesses)
__host__ __device__ __forceinline__ int tile2d_half(int L) { return ((L >> 1) + 1) & ~1; }
__host__ __device__ __forceinline__ int tile2d_groups(int L) { return (L + 3) >> 2; }  // items per row

enum { T2_FAST = 0, T2_GENERAL = 1, T2_OPEN = 2 };

// Accepted levels k of one compact table (see sys_table::base): the sites with count c < k flip.
__device__ __forceinline__ uint32_t accepted_levels(const sys_table &t, int tb, uint64_t g) {
  const uint32_t b = t.base[tb];
  uint32_t k = b;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) k += g < t.thr[tb][b + i < 7 ? b + i : 7] ? 1u : 0u;  // level 7 holds 0
  return k;
}
// bit b of k as a mask
__device__ __forceinline__ uint32_t bit_mask(uint32_t k, int b) { return (uint32_t)((int32_t)(k << (31 - b)) >> 31); }

// New spin word: flip where c < (spin ? k1 : k0), a bit-sliced compare (borrow chain).
constexpr int B3_NMAJ = 0x8E;  // majority(~a, b, c)
__device__ __forceinline__ uint64_t update_levels(uint32_t k0, uint32_t k1, const count3 &c, uint64_t si) {
  uint32_t r[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t s = (uint32_t)(si >> (32 * h));
    const uint32_t c0 = (uint32_t)(c.b0 >> (32 * h)), c1 = (uint32_t)(c.b1 >> (32 * h)), c2 = (uint32_t)(c.b2 >> (32 * h));
    uint32_t lt = ~c0 & b3<B3_MUX>(s, bit_mask(k1, 0), bit_mask(k0, 0));
    lt = b3<B3_NMAJ>(c1, b3<B3_MUX>(s, bit_mask(k1, 1), bit_mask(k0, 1)), lt);
    lt = b3<B3_NMAJ>(c2, b3<B3_MUX>(s, bit_mask(k1, 2), bit_mask(k0, 2)), lt);
    r[h] = s ^ lt;
  }
  return ((uint64_t)r[1] << 32) | r[0];
}

__device__ __forceinline__ void lds_ld2(const uint64_t *p, uint64_t &a, uint64_t &b) {
  const sa_v4u32 v = *reinterpret_cast<const sa_v4u32 *>(p);
  a = ((uint64_t)v.y << 32) | v.x;
  b = ((uint64_t)v.w << 32) | v.z;
}
__device__ __forceinline__ void lds_st2(uint64_t *p, uint64_t a, uint64_t b) {
  sa_v4u32 v;
  v.x = (uint32_t)a;
  v.y = (uint32_t)(a >> 32);
  v.z = (uint32_t)b;
  v.w = (uint32_t)(b >> 32);
  *reinterpret_cast<sa_v4u32 *>(p) = v;
}

// couplings of one colour's pair of an item
struct pair2d {
  uint64_t w0, e0, w1, e1, n0, n1, s0, s1;
};

// One tile of system `sys`, rows y0 - 2*ns .. y0 + th - 1 + 2*ns (WRAP: 0 .. L-1).
template <bool COUNTER, int MODE, int IT, bool WRAP>
__device__ __forceinline__ void tile2d(const tile2d_args &t, int sys, int band, uint64_t *lds) {
  const sweep_args &p = t.a;
  const int L = p.L, half = L >> 1, hp = tile2d_half(L), G = tile2d_groups(L), rowst = 2 * hp;
  const int halo = WRAP ? 0 : 2 * t.ns;
  const int R = WRAP ? L : t.th + 2 * halo;
  const int y0 = band * t.th;
  const uint64_t *s = p.s + (int64_t)sys * p.N;
  // items: row r, columns 4j .. 4j+3
  int r_[IT], j_[IT], y_[IT], reach[IT];
  bool two_[IT];  // the last group of a row with L % 4 == 2 has two columns, one site per colour
  pair2d J[IT][2];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int it = (int)threadIdx.x + i * (int)blockDim.x;
    const bool live = it < R * G;
    const int r = live ? it / G : 0, j = live ? it - r * G : 0;
    int y = y0 + r - halo;
    y = y < 0 ? y + L * ((L - 1 - y) / L) : y >= L ? y % L : y;
    r_[i] = r;
    j_[i] = j;
    y_[i] = y;
    // half-sweep h updates the rows with reach > h
    reach[i] = !live ? -1 : WRAP ? 0x7fffffff : min(r, R - 1 - r);
    const bool two = 4 * j + 2 < L;
    two_[i] = two;
    if (live) {
      const uint64_t *row = s + (int64_t)y * L + 4 * j;
      uint64_t a, b, c = 0, d = 0;
      a = row[0];
      b = row[1];
      if (two) {
        c = row[2];
        d = row[3];
      }
      lds_st2(lds + r * rowst + 2 * j, a, c);
      lds_st2(lds + r * rowst + hp + 2 * j, b, d);
      const int ys = y == L - 1 ? 0 : y + 1;
      const uint64_t *jx = p.jx + (int64_t)y * L, *jn = p.jy + (int64_t)y * L, *js = p.jy + (int64_t)ys * L;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int x = 4 * j + ((y + c) & 1), x2 = two ? x + 2 : x;
        pair2d &q = J[i][c];
        q.w0 = jx[x];
        q.e0 = jx[x == L - 1 ? 0 : x + 1];
        q.w1 = jx[x2];
        q.e1 = jx[x2 == L - 1 ? 0 : x2 + 1];
        q.n0 = jn[x];
        q.n1 = jn[x2];
        q.s0 = js[x];
        q.s1 = js[x2];
      }
    }
  }
  __syncthreads();
  for (int sw = 0; sw < t.ns; ++sw) {
    const sys_table &tab = p.tab[sys + sw * t.tab_step];
    const uint64_t *words = COUNTER ? nullptr : p.words + (int64_t)sw * p.N;
#pragma unroll
    for (int color = 0; color < 2; ++color) {
      const int h = 2 * sw + color;
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        if (reach[i] <= h) continue;
        const int r = r_[i], j = j_[i], y = y_[i];
        const int par = (y + color) & 1;
        const int rn = (WRAP && r == 0) ? L - 1 : r - 1, rs = (WRAP && r == L - 1) ? 0 : r + 1;
        uint64_t *own = lds + r * rowst + (par ? hp : 0);
        const uint64_t *oth = lds + r * rowst + (par ? 0 : hp);
        const uint64_t *nth = lds + rn * rowst + (par ? hp : 0), *sth = lds + rs * rowst + (par ? hp : 0);
        uint64_t a0, a1, m0, m1, n0, n1, s0, s1;
        lds_ld2(own + 2 * j, a0, a1);
        lds_ld2(oth + 2 * j, m0, m1);  // par 0: east of the first, of the second; par 1: west of them
        lds_ld2(nth + 2 * j, n0, n1);
        lds_ld2(sth + 2 * j, s0, s1);
        const bool two = two_[i];
        // the third x neighbour: par 0 the word west of the first site, par 1 east of the last
        const int kl = 2 * j + (two ? 2 : 1);
        const uint64_t far = oth[par ? (kl == half ? 0 : kl) : (j == 0 ? half - 1 : 2 * j - 1)];
        const uint64_t w0 = par ? m0 : far, e0 = par ? (two ? m1 : far) : m0;
        const uint64_t w1 = par ? m1 : m0, e1 = par ? far : m1;
        const pair2d &q = J[i][color];
        uint64_t g0, g1;
        if (COUNTER) {
          const u32x4 blk = counter_block((uint32_t)(4 * j + par + L * y), p.seed, p.sweep + (uint64_t)sw);
          g0 = counter_half(blk, 0);
          g1 = counter_half(blk, 1);
        } else {
          const int64_t rank = (int64_t)color * (p.N >> 1) + (int64_t)y * half + 2 * j;
          g0 = words[rank];
          g1 = two ? words[rank + 1] : 0;
        }
        uint64_t bw0 = xor3(q.w0, a0, w0), be1 = xor3(q.e1, a1, e1), be0 = xor3(q.e0, a0, e0);
        const bool west = MODE == T2_OPEN && !par && j == 0;          // the first site is x = 0
        const bool east = MODE == T2_OPEN && par && 4 * j + 4 >= L;   // the last site is x = L-1
        if (MODE == T2_OPEN) {  // missing open-x bond counts as satisfied (src/cpu_2dp.cpp:338-339)
          if (west) bw0 = ~0ULL;
          if (east && two) be1 = ~0ULL;
          if (east && !two) be0 = ~0ULL;
        }
        const count3 c0 = count4(bw0, be0, xor3(q.n0, a0, n0), xor3(q.s0, a0, s0));
        const count3 c1 = count4(xor3(q.w1, a1, w1), be1, xor3(q.n1, a1, n1), xor3(q.s1, a1, s1));
        uint64_t u0, u1;
        if (MODE == T2_FAST) {
          u0 = update_fast2(tab, g0, c0, a0);
          u1 = update_fast2(tab, g1, c1, a1);
        } else {
          uint32_t k00 = accepted_levels(tab, 0, g0), k01 = accepted_levels(tab, 1, g0);
          uint32_t k10 = accepted_levels(tab, 0, g1), k11 = accepted_levels(tab, 1, g1);
          if (MODE == T2_OPEN) {
            if (west || (east && !two)) {
              k00 = accepted_levels(tab, 2, g0);
              k01 = accepted_levels(tab, 3, g0);
            }
            if (east && two) {
              k10 = accepted_levels(tab, 2, g1);
              k11 = accepted_levels(tab, 3, g1);
            }
          }
          u0 = update_levels(k00, k01, c0, a0);
          u1 = update_levels(k10, k11, c1, a1);
        }
        lds_st2(own + 2 * j, u0, u1);  // a one-site item's second word is padding
      }
      __syncthreads();
    }
  }
  uint64_t *out = (WRAP ? p.s : t.out) + (int64_t)sys * p.N;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int r = r_[i], j = j_[i];
    // bands: the middle rows that exist (the last band may be shorter)
    const bool mine = reach[i] >= 0 && (WRAP || (r >= halo && r < R - halo && y0 + r - halo < L));
    if (!mine) continue;
    uint64_t a, b, c, d;
    lds_ld2(lds + r * rowst + 2 * j, a, c);
    lds_ld2(lds + r * rowst + hp + 2 * j, b, d);
    uint64_t *row = out + (int64_t)y_[i] * L + 4 * j;
    row[0] = a;
    row[1] = b;
    if (two_[i]) {
      row[2] = c;
      row[3] = d;
    }
  }
}

// ---- odd sides: the whole lattice in LDS, rows of L words.  The wrap neighbours in x and in y
// share a colour: the last column reads the new first one, the last row the new first one, and
// the corner both (row-major visits, src/cpu_2dp.cpp:106-114).  So a colour is updated in stages
// with a barrier after each: every site off the last column and row, then those on one of them,
// then the corner (colour 0).  In place: a stage reads old what later stages update.
//
// A thread owns IT items as above; the last item of a row has one column or three.  Bound by
// the update's chain and the five stages' barriers; what the random word accepts is formed in
// the first stage only (in each stage: general tables 9.7 instead of 7.8 us per sweep at L=89).
// Us per sweep, two launches with a thread per wrap group / here: L=17 x24 7.6 / 1.8, L=63 x1
// 7.6 / 3.1, L=89 x24 8.7 / 6.8, x1024 79 / 24.5, with a field x1 11.8 / 7.8; open x L=63 x8
// 14.1 / 7.4, L=89 x24 15.0 / 13.0.  In a batch the half-sweeps of many odd instances fill the
// chip together (52 instances of L 17..89: 10.0 us per sweep, as tiles 10.4), so it keeps them.
template <bool COUNTER, int MODE, int IT>
__device__ __forceinline__ void tile2d_odd(const tile2d_args &t, int sys, uint64_t *lds) {
  const sweep_args &p = t.a;
  const int L = p.L, G = tile2d_groups(L);
  uint64_t *s = p.s + (int64_t)sys * p.N;
  int j_[IT], y_[IT];
  pair2d J[IT][2];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int it = (int)threadIdx.x + i * (int)blockDim.x;
    const bool live = it < L * G;
    const int y = live ? it / G : 0, j = live ? it - y * G : 0;
    j_[i] = live ? j : -1;
    y_[i] = y;
    if (live) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (4 * j + c < L) lds[y * L + 4 * j + c] = s[(int64_t)y * L + 4 * j + c];
      const uint64_t *jx = p.jx + (int64_t)y * L, *jn = p.jy + (int64_t)y * L;
      const uint64_t *js = p.jy + (int64_t)(y == L - 1 ? 0 : y + 1) * L;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int x = min(4 * j + ((y + c) & 1), L - 1), x2 = min(x + 2, L - 1);  // beyond the row: not used
        pair2d &q = J[i][c];
        q.w0 = jx[x];
        q.e0 = jx[x == L - 1 ? 0 : x + 1];
        q.w1 = jx[x2];
        q.e1 = jx[x2 == L - 1 ? 0 : x2 + 1];
        q.n0 = jn[x];
        q.n1 = jn[x2];
        q.s0 = js[x];
        q.s1 = js[x2];
      }
    }
  }
  __syncthreads();
  for (int sw = 0; sw < t.ns; ++sw) {
    const sys_table &tab = p.tab[sys + sw * t.tab_step];
    const uint64_t *words = COUNTER ? nullptr : p.words + (int64_t)sw * p.N;
    // what a site's random word accepts, formed in the first stage, which every wave is in
    // (the levels of spin bit 0 | spin bit 1 << 8; FAST: bit 0 level 3, bit 1 level 4)
    auto levels = [&](int x, uint64_t g) {
      if (MODE == T2_FAST) return (g < tab.thr[0][3] ? 1u : 0u) | (g < tab.thr[0][4] ? 2u : 0u);
      uint32_t k0 = accepted_levels(tab, 0, g), k1 = accepted_levels(tab, 1, g);
      if (MODE == T2_OPEN && (x == 0 || x == L - 1)) {
        k0 = accepted_levels(tab, 2, g);
        k1 = accepted_levels(tab, 3, g);
      }
      return k0 | k1 << 8;
    };
    auto site = [&](int x, int y, uint64_t jw, uint64_t je, uint64_t jn, uint64_t js, uint32_t k) {
      uint64_t *row = lds + y * L;
      const uint64_t si = row[x];
      uint64_t bw = xor3(jw, si, row[x == 0 ? L - 1 : x - 1]), be = xor3(je, si, row[x == L - 1 ? 0 : x + 1]);
      if (MODE == T2_OPEN) {  // missing open-x bond counts as satisfied (src/cpu_2dp.cpp:338-339)
        if (x == 0) bw = ~0ULL;
        if (x == L - 1) be = ~0ULL;
      }
      const uint64_t un = lds[(y == 0 ? L - 1 : y - 1) * L + x], us = lds[(y == L - 1 ? 0 : y + 1) * L + x];
      const count3 c = count4(bw, be, xor3(jn, si, un), xor3(js, si, us));
      if (MODE == T2_FAST) row[x] = si ^ sel(c.b2, lvl(k & 2), ~(c.b1 & c.b0) | lvl(k & 1));
      else row[x] = update_levels(k & 255, k >> 8, c, si);
    };
#pragma unroll
    for (int color = 0; color < 2; ++color) {
      uint32_t k0[IT], k1[IT];
      // 0: off the last column and row, 1: on one of them, 2: the corner
      auto stage_of = [&](int x, int y) { return (x == L - 1 ? 1 : 0) + (y == L - 1 ? 1 : 0); };
#pragma unroll
      for (int st = 0; st < 3 - color; ++st) {
#pragma unroll
        for (int i = 0; i < IT; ++i) {
          const int j = j_[i], y = y_[i];
          if (j < 0) continue;
          const int x = 4 * j + ((y + color) & 1), x2 = x + 2;
          if (st == 0) {
            if (COUNTER) {
              const u32x4 blk = counter_block((uint32_t)(x + L * y), p.seed, p.sweep + (uint64_t)sw);
              k0[i] = levels(x, counter_half(blk, 0));
              k1[i] = levels(x2, counter_half(blk, 1));
            } else {
              const int64_t rank = x < L ? odd_rank(L, 1, color, x, y, 0) : 0;
              k0[i] = levels(x, words[rank]);
              k1[i] = levels(x2, x2 < L ? words[rank + 1] : 0);
            }
          }
          const pair2d &q = J[i][color];
          if (x < L && stage_of(x, y) == st) site(x, y, q.w0, q.e0, q.n0, q.s0, k0[i]);
          if (x2 < L && stage_of(x2, y) == st) site(x2, y, q.w1, q.e1, q.n1, q.s1, k1[i]);
        }
        __syncthreads();
      }
    }
  }
#pragma unroll
  for (int i = 0; i < IT; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (j_[i] >= 0 && 4 * j_[i] + c < L) s[(int64_t)y_[i] * L + 4 * j_[i] + c] = lds[y_[i] * L + 4 * j_[i] + c];
}

template <bool COUNTER, int MODE, int IT>
__global__ void __launch_bounds__(1024) k_tile2d_odd(tile2d_args t) {
  extern __shared__ __align__(16) uint64_t lds[];
  tile2d_odd<COUNTER, MODE, IT>(t, (int)blockIdx.x, lds);
}

template <bool COUNTER, int MODE, int IT, bool WRAP>
__global__ void __launch_bounds__(1024) k_tile2d(tile2d_args t) {
  extern __shared__ __align__(16) uint64_t lds[];
  const int sys = (int)blockIdx.x / t.bands;
  tile2d<COUNTER, MODE, IT, WRAP>(t, sys, (int)blockIdx.x - sys * t.bands, lds);
}

}  // namespace sa
