// sa_tile3d.hpp -- one 3D sweep (both colours) per launch, tiles of columns in LDS.
//
// A ladder too small to fill the chip with column walks is bound by latency: two launches
// per sweep, each one dependent chain of loads, arithmetic and stores.  Here a workgroup
// owns a tile of tx x ty columns (full z) of one system, loads it with a halo of two
// columns on every side into LDS, updates colour 0 on the tile and one halo column around
// it (the same words the neighbouring tiles compute), then colour 1 on the tile, and
// writes the tile to the other spin array, so no workgroup waits for another and the sweep
// is one launch.  A lattice that fits LDS whole (WHOLE: no halo, wrapping indices) is kept
// there for `ns` sweeps.
//
// The z walk is a scan, as in k_sweep3d_zscan: a column is cut into G segments of S planes,
// lane = column * 2^lg + segment (2^lg >= G, the rest idle); the new word of a plane is a
// per-lane map (f0, f1) of the new word below it.  The count of the five bonds that do not point down is formed once,
// the two outcomes are two cheap selects of it.  The last of the four-plane segments may be
// shorter (its missing planes are identity maps), so any even L up to 256 is served, and odd
// ones in the form further down.
//
// Everything a segment reads lies along z: the ladder keeps a copy of its couplings with z
// fastest, made when the couplings are set and first needed, and LDS holds columns.  A
// wave's coupling load is then 512 B or 1 KB in a row (with x fastest, every lane touched a
// cache line of its own, and the address unit took 9 of a sweep's 22 thousand cycles for
// them), and both planes of a segment are one 128-bit access.
//
// One L=64 system: 12.6 -> 7.2 us per sweep (kernel trace: 6.0 at least); 16 systems of L=32
// 15.6 -> 7.4; 12 of L=16, held whole, 9.5 -> 2.9; 8 of L=48 with a field 37 -> 19.5.
#pragma once

#include <algorithm>

#include "sa_kernels.hpp"
#include "sa_tile2d.hpp"
#include "sa_tile_place.hpp"

namespace sa {

struct tile3d_args {
  sweep_args a;
  uint64_t *out;     // written spin array (WHOLE: a.s itself)
  int tx, ty;        // columns of a tile (WHOLE: L, L)
  int ntx, nty;      // tiles per side
  int G, C, lg;      // segments per column, columns per wave, log2 of the lanes per column
  int lp;            // LDS words per column (even, 2 modulo 4)
  const uint64_t *jxt, *jyt, *jzt;  // couplings with z fastest: word (x + L*y) * L + z
  int chunks0, chunks1;  // waves' worth of columns of colour 0 / 1
  int recip_n0, recip_n1, recip_pairs, recip_hw, recip_ntx;  // ceil(2^20 / d): columns per row of colour 0 / 1, pairs of a plane, pairs of a row, tiles of a row
  uint32_t recip_per;  // tile_recip(tiles of a system)
  int zstep;         // planes the block's threads load at a time
  int ns;            // sweeps (1 unless WHOLE)
  int64_t tab_step;  // tables per sweep
};

__host__ __device__ __forceinline__ int column_stride(int L);
__host__ __device__ __forceinline__ int odd_list_words(int W, int H);

// The geometry part of the arguments for a tile of tx x ty columns (whole: L x L), S planes
// per segment and blocks of `threads`; chunks0 / chunks1 are set too.  Returns the LDS bytes,
// 0 where the form does not apply.
inline size_t tile3d_setup(tile3d_args &a, int L, bool whole, int tx, int ty, int S, int threads) {
  const bool odd = L & 1;
  a.tx = whole ? L : tx;
  a.ty = whole ? L : ty;
  const int W = whole ? L : tx + 4, H = whole ? L : ty + 4;
  if (!whole && (tx > L || ty > L || (odd && (W > L || H > L)))) return 0;
  a.ntx = (L + a.tx - 1) / a.tx;
  a.nty = (L + a.ty - 1) / a.ty;
  a.G = (L + S - 1) / S;
  if (a.G < 2 || a.G > 64) return 0;
  a.lg = 1;
  while ((1 << a.lg) < a.G) ++a.lg;
  a.C = 64 >> a.lg;
  a.lp = column_stride(L) % 4 == 0 ? column_stride(L) + 2 : column_stride(L);
  // odd sides: one more column per row at most
  const int col0 = whole ? (L * L + 1) / 2 : (tx / 2 + 1) * (ty + 2), col1 = whole ? L * L / 2 : tx / 2 * ty;
  a.chunks0 = (col0 + a.C - 1) / a.C;
  a.chunks1 = (col1 + a.C - 1) / a.C;
  const int row = odd ? W : W / 2;  // columns or pairs of columns a thread loads
  if (row * H > threads) return 0;
  a.zstep = threads / (row * H);
  a.recip_pairs = small_recip(row * H);
  a.recip_hw = small_recip(row);
  a.recip_ntx = small_recip(a.ntx);
  a.recip_per = tile_recip((uint32_t)(a.ntx * a.nty));
  a.recip_n0 = small_recip(whole ? std::max(L / 2, 1) : tx / 2 + 1);
  a.recip_n1 = small_recip(whole ? std::max(L / 2, 1) : tx / 2);
  return ((size_t)W * H * a.lp + (odd ? odd_list_words(W, H) : 0)) * 8;
}

// the two outcomes of a site's update as functions of the bond below it
struct flips {
  uint64_t f0, f1;  // flip when that bond is unsatisfied / satisfied
};

// FAST: levels 0..3 always accept, a4 >= a5 >= a6 (masks); (p2 p1 p0) = satisfied among five
__device__ __forceinline__ flips flips_fast(uint32_t a4, uint32_t a5, uint32_t a6, uint64_t p0, uint64_t p1, uint64_t p2) {
  uint32_t r0[2], r1[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t q0 = (uint32_t)(p0 >> (32 * h)), q1 = (uint32_t)(p1 >> (32 * h)), q2 = (uint32_t)(p2 >> (32 * h));
    // p <= 3: accept; 4: a4; 5: a5
    r0[h] = ~q2 | b3<B3_MUX>(q0, a5, a4);
    // p + 1 <= 3: accept; 4: a4; 5: a5; 6: a6
    r1[h] = b3<B3_MUX>(q2, b3<B3_MUX>(q0, a6, a5), ~(q1 & q0) | a4);
  }
  return flips{((uint64_t)r0[1] << 32) | r0[0], ((uint64_t)r1[1] << 32) | r1[0]};
}
// general compact tables: k0 / k1 accepted levels for spin bit 0 / 1
__device__ __forceinline__ uint64_t less_levels(uint32_t k0, uint32_t k1, uint64_t p0, uint64_t p1, uint64_t p2, uint64_t si) {
  return update_levels(k0, k1, count3{p0, p1, p2}, si) ^ si;
}
__device__ __forceinline__ flips flips_general(uint32_t k0, uint32_t k1, uint64_t p0, uint64_t p1, uint64_t p2, uint64_t si) {
  const uint32_t l0 = k0 ? k0 - 1 : 0, l1 = k1 ? k1 - 1 : 0;  // p + 1 < k
  return flips{less_levels(k0, k1, p0, p1, p2, si), less_levels(l0, l1, p0, p1, p2, si)};
}

__device__ __forceinline__ uint64_t ld_off(const uint64_t *p, uint32_t byte_off) {
  return *reinterpret_cast<const uint64_t *>(reinterpret_cast<const char *>(p) + byte_off);
}

// A lane's column segment of one colour: where its words lie.
struct seg3d {
  int z0, g, base;        // first plane, segment, lane of the column's segment 0
  bool live;              // false: an idle lane (reads a valid column, writes nothing)
  uint32_t c0, ce, cs;    // columns x + L*y: the site's, its +x and its +y neighbour's
  int k, kw, ke, kn, ks;  // LDS columns: the site's, its four in-plane neighbours'
  int64_t rank;           // replay word of the column's plane 0
  uint32_t rstep;         // replay words of this colour per plane
};
template <int S>
struct seg3d_couplings {
  uint64_t jw[S], je[S], jn[S], js[S], jd[S], ju;  // -x, +x, -y, +y, +z bonds; the first plane's -z bond
};

// wave `chunk`'s columns of one colour; LDS column row * W/2 + i of a colour is pair column
// i of a row (tx = 2i + ((row + colour) & 1))
template <int S, bool WHOLE>
__device__ __forceinline__ seg3d tile3d_segment(const tile3d_args &t, int color, int chunk, int ox, int oy) {
  seg3d q;
  const int L = t.a.L, hw = WHOLE ? L >> 1 : (t.tx >> 1) + 2;
  const int nI = WHOLE ? L >> 1 : (t.tx >> 1) + (color == 0 ? 1 : 0);
  const int r0 = WHOLE ? 0 : (color == 0 ? 1 : 2), nrows = WHOLE ? L : (color == 0 ? t.ty + 2 : t.ty);
  const int ncol = nI * nrows, lane = (int)threadIdx.x & 63;
  const int cc = lane >> t.lg;
  q.base = cc << t.lg;
  q.g = lane - q.base;
  q.z0 = q.g < t.G ? q.g * S : 0;
  const int col = chunk * t.C + cc;
  q.live = q.g < t.G && col < ncol;
  const int cl = q.live ? col : 0;
  const int row = small_div(cl, color == 0 ? t.recip_n0 : t.recip_n1), idx = cl - row * nI, ty = r0 + row;
  const int P = (ty + color) & 1;
  const int i = WHOLE ? idx : idx + (color == 0 ? 1 - P : 1);
  int x = WHOLE ? 2 * i + P : ox + 2 * i + P, y = WHOLE ? ty : oy + ty;
  if (!WHOLE) {  // -2 <= x, y < 2L
    x = x < 0 ? x + L : x >= L ? x - L : x;
    y = y < 0 ? y + L : y >= L ? y - L : y;
  }
  q.c0 = (uint32_t)(x + L * y);
  q.ce = (uint32_t)((x == L - 1 ? 0 : x + 1) + L * y);
  q.cs = (uint32_t)(x + L * (y == L - 1 ? 0 : y + 1));
  const int k = ty * hw + i;
  q.k = k;
  if (WHOLE) {
    q.kw = P ? k : (i == 0 ? k + hw - 1 : k - 1);
    q.ke = P ? (i == hw - 1 ? k - hw + 1 : k + 1) : k;
    q.kn = ty == 0 ? k + (L - 1) * hw : k - hw;
    q.ks = ty == L - 1 ? k - (L - 1) * hw : k + hw;
  } else {
    q.kw = P ? k : k - 1;
    q.ke = P ? k + 1 : k;
    q.kn = k - hw;
    q.ks = k + hw;
  }
  q.rank = (int64_t)color * (t.a.N >> 1) + (int64_t)y * (L >> 1) + (x >> 1);
  q.rstep = (uint32_t)(L * L) >> 1;
  return q;
}

// words per column of the couplings with z fastest: even, so that pairs of planes are 16 bytes
__host__ __device__ __forceinline__ int column_stride(int L) { return (L + 1) & ~1; }

// S words of a column from plane z0 on, 16 bytes at a time (z0 even; beyond the lattice, in
// a short last segment, the last pair of planes again; an odd side's last pair ends in padding)
template <int S>
__device__ __forceinline__ void column_words(const uint64_t *p, uint32_t col, int z0, int L, uint64_t (&w)[S]) {
  const uint32_t st = (uint32_t)column_stride(L);
#pragma unroll
  for (int j = 0; j < S; j += 2) {
    const uint64_t *q = reinterpret_cast<const uint64_t *>(
        reinterpret_cast<const char *>(p) + (col * st + (uint32_t)min(z0 + j, (L - 1) & ~1)) * 8u);
    lds_ld2(q, w[j], w[j + 1]);
  }
}

template <int S>
__device__ __forceinline__ void tile3d_load(const tile3d_args &t, const seg3d &q, seg3d_couplings<S> &d) {
  const int L = t.a.L;
  uint64_t jz[S];
  column_words<S>(t.jxt, q.c0, q.z0, L, d.jw);
  column_words<S>(t.jxt, q.ce, q.z0, L, d.je);
  column_words<S>(t.jyt, q.c0, q.z0, L, d.jn);
  column_words<S>(t.jyt, q.cs, q.z0, L, d.js);
  column_words<S>(t.jzt, q.c0, q.z0, L, jz);
  const int zn = q.z0 + S;  // the plane above the segment; above the lattice's last, plane 0
  const uint64_t jn = ld_off(t.jzt, (q.c0 * (uint32_t)column_stride(L) + (uint32_t)(zn >= L ? 0 : zn)) * 8u);
  d.ju = jz[0];
#pragma unroll
  for (int j = 0; j < S; ++j) d.jd[j] = (j == S - 1 || q.z0 + j + 1 >= L) ? jn : jz[j + 1 < S ? j + 1 : j];
}

// the segment's random words
template <bool COUNTER, int S>
__device__ __forceinline__ void tile3d_random(const tile3d_args &t, const uint64_t *words, uint64_t sweep, const seg3d &q,
                                              uint64_t (&g)[S]) {
  const uint32_t L2 = (uint32_t)(t.a.L * t.a.L);
  if (COUNTER) {
#pragma unroll
    for (int j = 0; j < S; j += 2) {
      const u32x4 blk = counter_block(q.c0 + (uint32_t)(q.z0 + j) * L2, t.a.seed, sweep);
      g[j] = counter_half(blk, 0);
      g[j + 1] = counter_half(blk, 1);
    }
  } else {
#pragma unroll
    for (int j = 0; j < S; ++j) g[j] = words[q.rank + (int64_t)min(q.z0 + j, t.a.L - 1) * q.rstep];
  }
}

// the map of the lane `d` (a power of two) below in the wave; within rows of 16 lanes for d < 16
template <int CTRL>
__device__ __forceinline__ uint64_t dpp64(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(v >> 32), (int)(v >> 32), CTRL, 0xf, 0xf, false);
  return ((uint64_t)hi << 32) | lo;
}
constexpr int kDppRowShr = 0x110, kDppWaveShr1 = 0x138, kDppBcast15 = 0x142, kDppBcast31 = 0x143;
template <int CTRL>
__device__ __forceinline__ void scan_step(zmap &M, bool take) {
  const zmap T{dpp64<CTRL>(M.f0), dpp64<CTRL>(M.f1)};
  const zmap R = zcompose(M, T);
  if (take) M = R;
}
// Inclusive scan over a column's 2^lg lanes with data-parallel-primitive moves (a lane
// shuffle goes through LDS and takes ten times as long): shifts within rows of 16 lanes,
// then the last lane of a row to the whole next row.
__device__ __forceinline__ void scan_columns(zmap &M, int g, int lg) {
  const int r = g & 15;
  scan_step<kDppRowShr + 1>(M, r >= 1);
  if (lg > 1) scan_step<kDppRowShr + 2>(M, r >= 2);
  if (lg > 2) scan_step<kDppRowShr + 4>(M, r >= 4);
  if (lg > 3) scan_step<kDppRowShr + 8>(M, r >= 8);
  if (lg > 4) scan_step<kDppBcast15>(M, (g & 16) != 0);
  if (lg > 5) scan_step<kDppBcast31>(M, (g & 32) != 0);
}

// The colour's update of a segment; A / O: the LDS columns of this colour and the other
// (ODD: all columns, A == O).
template <bool FAST, int S, bool ODD = false>
__device__ __forceinline__ void tile3d_update(const tile3d_args &t, const sys_table &tab, const uint64_t (&g64)[S],
                                              const seg3d &q, const seg3d_couplings<S> &d, uint64_t *A,
                                              const uint64_t *O) {
  const int L = t.a.L, lp = t.lp, z0 = q.z0;
  uint64_t si[S + 1], nw[S], ne[S], nn[S], ns[S];
#pragma unroll
  for (int j = 0; j < S; j += 2) {
    const int z = min(z0 + j, (L - 1) & ~1);
    lds_ld2(A + q.k * lp + z, si[j], si[j + 1]);
    lds_ld2(O + q.kw * lp + z, nw[j], nw[j + 1]);
    lds_ld2(O + q.ke * lp + z, ne[j], ne[j + 1]);
    lds_ld2(O + q.kn * lp + z, nn[j], nn[j + 1]);
    lds_ld2(O + q.ks * lp + z, ns[j], ns[j + 1]);
  }
  si[S] = A[q.k * lp + (z0 + S >= L ? 0 : z0 + S)];
  const uint64_t up0 = A[q.k * lp + L - 1];  // old plane L-1: plane 0's word below
  zmap F[S];
  uint64_t new0 = 0;
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const uint64_t s = si[j];
    const uint64_t qw = xor3(d.jw[j], s, nw[j]), qe = xor3(d.je[j], s, ne[j]);
    const uint64_t qn = xor3(d.jn[j], s, nn[j]), qs = xor3(d.js[j], s, ns[j]);
    const uint64_t s1 = xor3(qw, qe, qn), k1 = maj3(qw, qe, qn);
    // bond below with an all-0 word below; plane 0 has the old plane L-1 there
    const uint64_t ju = j == 0 ? d.ju : d.jd[j - 1];
    const uint64_t b = xor3(ju, s, (j == 0 && z0 == 0) ? up0 : 0);
    // the plane's map with the word dn above it
    auto map = [&](uint64_t dn) {
      const uint64_t qd = xor3(d.jd[j], s, dn);
      const uint64_t p0 = xor3(qs, qd, s1), k2 = maj3(qs, qd, s1);
      const uint64_t p1 = k1 ^ k2, p2 = k1 & k2;
      flips f;
      if (FAST) {
        const uint32_t a4 = g64[j] < tab.thr[0][4] ? ~0u : 0u, a5 = g64[j] < tab.thr[0][5] ? ~0u : 0u;
        const uint32_t a6 = g64[j] < tab.thr[0][6] ? ~0u : 0u;
        f = flips_fast(a4, a5, a6, p0, p1, p2);
      } else {
        f = flips_general(accepted_levels(tab, 0, g64[j]), accepted_levels(tab, 1, g64[j]), p0, p1, p2, s);
      }
      F[j].f0 = s ^ sel(b, f.f1, f.f0);
      F[j].f1 = s ^ sel(b, f.f0, f.f1);
    };
    // plane L-1 sees the new plane 0 above it
    map(j > 0 && z0 + j == L - 1 ? new0 : si[j + 1]);
    if (j == 0) {
      if (z0 == 0) F[0].f1 = F[0].f0;
      new0 = shfl64(F[0].f0, q.base);  // segment 0 of this column
      if (ODD && z0 == L - 1) map(new0);  // a last segment of one plane
    }
    if ((ODD || S > 2) && z0 + j >= L) F[j] = zmap{0, ~0ULL};  // no such plane
  }
  zmap M = F[0];
#pragma unroll
  for (int j = 1; j < S; ++j) M = zcompose(F[j], M);
  scan_columns(M, q.g, t.lg);
  const uint64_t below = dpp64<kDppWaveShr1>(M.f0);  // the new word below the segment's first plane
  if (q.live) {
    uint64_t v = below;
#pragma unroll
    for (int j = 0; j < S; j += 2) {
      const uint64_t v0 = (j == 0 && z0 == 0) ? F[0].f0 : sel(v, F[j].f1, F[j].f0);
      v = sel(v0, F[j + 1].f1, F[j + 1].f0);
      if (S == 2 || z0 + j < L) lds_st2(A + q.k * lp + z0 + j, v0, v);  // ODD: plane L is padding
    }
  }
}

// Tile (bx, by) of system sys.  ONE: a wave has at most one chunk of columns per colour,
// whose places and couplings it then keeps: colour 0's couplings are in flight while the tile
// is loaded, colour 1's while colour 0 is updated, and with several sweeps both are loaded once.
template <bool COUNTER, bool FAST, int S, bool WHOLE, bool ONE>
__device__ __forceinline__ void tile3d(const tile3d_args &t, int sys, int bx, int by, uint64_t *lds) {
  const sweep_args &p = t.a;
  const int L = p.L, W = WHOLE ? L : t.tx + 4, H = WHOLE ? L : t.ty + 4, hw = W >> 1, lp = t.lp;
  const int ox = WHOLE ? 0 : bx * t.tx - 2, oy = WHOLE ? 0 : by * t.ty - 2;
  uint64_t *pl[2] = {lds, lds + H * hw * lp};  // LDS columns of the two colours
  const uint64_t *s = p.s + (int64_t)sys * p.N;
  const int pairs = H * hw, L2 = L * L, wv = (int)threadIdx.x >> 6, nw = (int)blockDim.x >> 6;
  // tile and halo into LDS, colours apart: a thread keeps one pair of a plane, four planes in flight
  const int zt = small_div((int)threadIdx.x, t.recip_pairs), zstep = t.zstep;  // zstep * pairs <= blockDim.x
  const int k = (int)threadIdx.x - zt * pairs, ty = small_div(k, t.recip_hw);
  int x = ox + 2 * (k - ty * hw), y = oy + ty;
  x = x < 0 ? x + L : x >= L ? x - L : x;
  y = y < 0 ? y + L : y >= L ? y - L : y;
  const uint64_t *col = s + (y * L + x);
  auto fetch = [&](int zb, uint64_t (&a)[4], uint64_t (&b)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) lds_ld2(col + (int64_t)min(zb + u * zstep, L - 1) * L2, a[u], b[u]);
  };
  auto put = [&](int zb, const uint64_t (&a)[4], const uint64_t (&b)[4]) {
    if (zt >= zstep) return;
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // beyond the last plane: the last plane's words again
      const int at = k * lp + min(zb + u * zstep, L - 1);
      pl[0][at] = (ty & 1) ? b[u] : a[u];
      pl[1][at] = (ty & 1) ? a[u] : b[u];
    }
  };
  seg3d q0, q1;  // a wave beyond the last chunk is idle (reads valid columns)
  seg3d_couplings<S> d0, d1;
  uint64_t g0[S], g1[S];
  {
    uint64_t a[4], b[4];
    fetch(zt, a, b);
    if (ONE) {  // while they are on their way: both colours' places and random words, colour 0's couplings
      q0 = tile3d_segment<S, WHOLE>(t, 0, wv, ox, oy);
      tile3d_load<S>(t, q0, d0);
      q1 = tile3d_segment<S, WHOLE>(t, 1, wv, ox, oy);
      if (!WHOLE) {
        tile3d_random<COUNTER, S>(t, p.words, p.sweep, q0, g0);
        tile3d_random<COUNTER, S>(t, p.words, p.sweep, q1, g1);
      }
    }
    put(zt, a, b);
    for (int zb = zt + 4 * zstep; zb < L; zb += 4 * zstep) {
      fetch(zb, a, b);
      put(zb, a, b);
    }
  }
  __syncthreads();
  if (ONE) tile3d_load<S>(t, q1, d1);
  for (int sw = 0; sw < (WHOLE ? t.ns : 1); ++sw) {
    const sys_table &tab = p.tab[sys + sw * t.tab_step];
    const uint64_t *words = COUNTER ? nullptr : p.words + (int64_t)sw * p.N;
    const uint64_t sweep = p.sweep + (uint64_t)sw;
    if (ONE) {
      if (wv < t.chunks0) {
        if (WHOLE) tile3d_random<COUNTER, S>(t, words, sweep, q0, g0);
        tile3d_update<FAST, S>(t, tab, g0, q0, d0, pl[0], pl[1]);
      }
      __syncthreads();
      if (wv < t.chunks1) {
        if (WHOLE) tile3d_random<COUNTER, S>(t, words, sweep, q1, g1);
        tile3d_update<FAST, S>(t, tab, g1, q1, d1, pl[1], pl[0]);
      }
      __syncthreads();
    } else {
#pragma unroll 1
      for (int c = 0; c < 2; ++c) {
        for (int ch = wv; ch < (c ? t.chunks1 : t.chunks0); ch += nw) {
          const seg3d q = tile3d_segment<S, WHOLE>(t, c, ch, ox, oy);
          seg3d_couplings<S> d;
          uint64_t g[S];
          tile3d_load<S>(t, q, d);
          tile3d_random<COUNTER, S>(t, words, sweep, q, g);
          tile3d_update<FAST, S>(t, tab, g, q, d, lds + c * H * hw * lp, lds + (1 - c) * H * hw * lp);
        }
        __syncthreads();
      }
    }
  }
  // the tile's own columns: the threads that loaded them
  const int i = k - ty * hw;
  const bool mine = zt < zstep && (WHOLE || (i >= 1 && i <= t.tx >> 1 && ty >= 2 && ty < t.ty + 2 && ox + 2 * i < L &&
                                             oy + ty < L));  // not beyond the lattice in a shorter last tile
  if (mine) {
    uint64_t *out = (WHOLE ? p.s : t.out) + (int64_t)sys * p.N + (y * L + x);
    for (int z = zt; z < L; z += zstep) {
      const uint64_t e = pl[0][k * lp + z], o = pl[1][k * lp + z];
      lds_st2(out + (int64_t)z * L2, (ty & 1) ? o : e, (ty & 1) ? e : o);
    }
  }
}

// ---------------------------------------------------------------- odd sides
// With odd L the sites x = L-1 and x = 0 of a row have the same colour, and so have y = L-1
// and y = 0: in a half-sweep (L-1, y) sees the new word of (0, y) in its plane, (x, L-1) that
// of (x, 0), and the corner (L-1, L-1), of colour 0, those of (0, L-1) and (L-1, 0); all other
// same-colour neighbours across the wrap are seen old (the reference's row-major order,
// src/cpu_3d.cpp:94-105).  So a colour is updated in stages, each whole columns with a
// barrier after it: first every column off the last column and row, then those on one of
// them, then the corner.  In place, a stage reads old what later stages update.
// The tiles' grid is shifted by two columns so that both wraps lie inside tile 0's own
// columns, two away from its edge; every other tile is an ordinary one.  A tile is at most
// L-4 wide, so no column occurs in it twice.  LDS keeps all columns in one array, and each
// block first lists its columns by colour and stage.  Each stage costs its latency, about
// 0.8 us; 12 systems of L=27: 50 -> 11 us per sweep, one of L=63 134 -> 12.
constexpr int kOddShift = 2;
constexpr int kOddPhases = 5;  // colour 0 stages 1, 2, 3; colour 1 stages 1, 2

// LDS words (64 bit) of the column lists: first stages, second stages, the corner
__host__ __device__ __forceinline__ int odd_list_cap(int W, int H, int phase) {
  return phase == 0 || phase == 3 ? H * (W / 2 + 1) : phase == 2 ? 4 : W + H;
}
__host__ __device__ __forceinline__ int odd_list_words(int W, int H) {
  int n = 0;
  for (int q = 0; q < kOddPhases; ++q) n += odd_list_cap(W, H, q);
  return (n + 3) / 4 + 4;  // 16-bit entries, five counters
}

template <bool COUNTER, bool FAST, int S, bool WHOLE>
__device__ __forceinline__ void tile3d_odd(const tile3d_args &t, int sys, int bx, int by, uint64_t *lds) {
  const sweep_args &p = t.a;
  const int L = p.L, W = WHOLE ? L : t.tx + 4, H = WHOLE ? L : t.ty + 4, lp = t.lp, ncols = W * H;
  const int cx = WHOLE ? L : min(t.tx, L - bx * t.tx), cy = WHOLE ? L : min(t.ty, L - by * t.ty);  // own columns
  const int ox = WHOLE ? 0 : bx * t.tx - kOddShift - 2, oy = WHOLE ? 0 : by * t.ty - kOddShift - 2;
  const int64_t L2 = (int64_t)L * L;
  auto wrap = [&](int v) { return v < 0 ? v + L : v >= L ? v - L : v; };
  uint64_t *A = lds;
  int *cnt = reinterpret_cast<int *>(lds + ncols * lp);
  uint16_t *list[kOddPhases];
  {
    uint16_t *q = reinterpret_cast<uint16_t *>(cnt + 8);
#pragma unroll
    for (int f = 0; f < kOddPhases; ++f) {
      list[f] = q;
      q += odd_list_cap(W, H, f);
    }
  }
  if (threadIdx.x < 8) cnt[threadIdx.x] = 0;
  __syncthreads();
  // a thread loads one column's planes zt, zt + zstep, ...
  const int zt = small_div((int)threadIdx.x, t.recip_pairs), zstep = t.zstep;
  const int k = (int)threadIdx.x - zt * ncols, ty = small_div(k, t.recip_hw), tx = k - ty * W;
  const int x = wrap(ox + tx), y = wrap(oy + ty);
  const uint64_t *col = p.s + (int64_t)sys * p.N + (y * L + x);
  for (int zb = zt; zb < L; zb += 8 * zstep) {
    uint64_t a[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = col[min(zb + u * zstep, L - 1) * L2];
    if (zb == zt && zt == 0) {  // each column once: into its colour's and stage's list
      const int c = (x + y) & 1, e = (c == 0 ? 1 : 2);
      const bool in = WHOLE || (tx >= e && tx < cx + 4 - e && ty >= e && ty < cy + 4 - e);
      if (in) {
        const int stage = (x == L - 1 ? 1 : 0) + (y == L - 1 ? 1 : 0), f = c == 0 ? stage : 3 + stage;
        list[0][(f == 0 ? 0 : f == 1 ? list[1] - list[0] : f == 2 ? list[2] - list[0] : f == 3 ? list[3] - list[0]
                                                                                               : list[4] - list[0]) +
                atomicAdd(&cnt[f], 1)] = (uint16_t)k;
      }
    }
    if (zt < zstep) {
#pragma unroll
      for (int u = 0; u < 8; ++u) A[k * lp + min(zb + u * zstep, L - 1)] = a[u];
    }
  }
  __syncthreads();
  const int lane = (int)threadIdx.x & 63, nw = (int)blockDim.x >> 6, cc = lane >> t.lg;
  for (int sw = 0; sw < (WHOLE ? t.ns : 1); ++sw) {
    const sys_table &tab = p.tab[sys + sw * t.tab_step];
    const uint64_t *words = COUNTER ? nullptr : p.words + (int64_t)sw * p.N;
    const uint64_t sweep = p.sweep + (uint64_t)sw;
    const uint16_t *cols = list[0];
#pragma unroll 1
    for (int f = 0; f < kOddPhases; ++f) {
      const int n = cnt[f], color = f < 3 ? 0 : 1;
      if (n == 0) {  // the same for the whole block
        cols += odd_list_cap(W, H, f);
        continue;
      }
      for (int ch = (int)threadIdx.x >> 6; ch * t.C < n; ch += nw) {
        seg3d q;
        q.base = cc << t.lg;
        q.g = lane - q.base;
        q.z0 = q.g < t.G ? q.g * S : 0;
        const int at = ch * t.C + cc;
        q.live = q.g < t.G && at < n;
        q.k = cols[at < n ? at : 0];
        const int qy = small_div(q.k, t.recip_hw), qx = q.k - qy * W;
        const int gx = wrap(ox + qx), gy = wrap(oy + qy);
        q.c0 = (uint32_t)(gx + L * gy);
        q.ce = (uint32_t)((gx == L - 1 ? 0 : gx + 1) + L * gy);
        q.cs = (uint32_t)(gx + L * (gy == L - 1 ? 0 : gy + 1));
        q.kw = WHOLE && qx == 0 ? q.k + L - 1 : q.k - 1;
        q.ke = WHOLE && qx == L - 1 ? q.k - (L - 1) : q.k + 1;
        q.kn = WHOLE && qy == 0 ? q.k + (L - 1) * W : q.k - W;
        q.ks = WHOLE && qy == L - 1 ? q.k - (L - 1) * W : q.k + W;
        if (!COUNTER) {
          q.rank = odd_rank(L, L, color, gx, gy, 0);
          q.rstep = (uint32_t)(color ? L2 / 2 : (L2 + 1) / 2);
        }
        seg3d_couplings<S> d;
        uint64_t g[S];
        tile3d_load<S>(t, q, d);
        tile3d_random<COUNTER, S>(t, words, sweep, q, g);
        tile3d_update<FAST, S, true>(t, tab, g, q, d, A, A);
      }
      cols += odd_list_cap(W, H, f);
      __syncthreads();
    }
  }
  if (zt < zstep && (WHOLE || (tx >= 2 && tx < cx + 2 && ty >= 2 && ty < cy + 2))) {
    uint64_t *out = (WHOLE ? p.s : t.out) + (int64_t)sys * p.N + (y * L + x);
    for (int z = zt; z < L; z += zstep) out[z * L2] = A[k * lp + z];
  }
}

template <bool COUNTER, bool FAST, int S, bool WHOLE>
__global__ void __launch_bounds__(1024) k_tile3d_odd(tile3d_args t) {
  extern __shared__ __align__(16) uint64_t lds[];
  const uint32_t per = (uint32_t)(t.ntx * t.nty);  // blocks to tiles as in k_tile3d
  const uint32_t b = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (b >= per * (uint32_t)t.a.nsys) return;
  const tile_place p = place_tile(b, per, t.recip_per, (uint32_t)t.ntx, t.recip_ntx);
  tile3d_odd<COUNTER, FAST, S, WHOLE>(t, (int)p.sys, (int)p.bx, (int)p.by, lds);
}

template <bool COUNTER, bool FAST, int S, bool WHOLE, bool ONE>
__global__ void __launch_bounds__(1024) k_tile3d(tile3d_args t) {
  extern __shared__ __align__(16) uint64_t lds[];
  // Blocks go round-robin over the 8 XCDs: give each XCD a contiguous range of tiles, whole
  // systems where there are several.  A system's words then stay in the L2 that wrote them,
  // halos and couplings included (3D L=32, 16 systems: 7.4 us per sweep; every XCD a part of
  // every system 8.4).
  const uint32_t per = (uint32_t)(t.ntx * t.nty);
  const uint32_t b = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (b >= per * (uint32_t)t.a.nsys) return;
  const tile_place p = place_tile(b, per, t.recip_per, (uint32_t)t.ntx, t.recip_ntx);
  tile3d<COUNTER, FAST, S, WHOLE, ONE>(t, (int)p.sys, (int)p.bx, (int)p.by, lds);
}

}  // namespace sa
