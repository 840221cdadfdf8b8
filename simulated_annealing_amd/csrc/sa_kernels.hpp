// sa_kernels.hpp -- gfx950 kernels of the multispin +-J Metropolis sweep.
//
// Data layout in HBM (one ladder = `nsys` systems of one geometry that share the
// couplings and the random stream, i.e. the temperatures of a parallel-tempering
// run or a single annealed system):
//   s   : nsys x N uint64 words, system-major, site i = x + L*y (+ L*L*z); bit k of
//         a word is lane k (64 independent disorder samples).
//   jx, jy, jz : N words each, deduplicated: jx[i] couples i to its -x neighbour,
//         jy[i] to -y, jz[i] to -z (the reference keeps each bond twice,
//         src/gpu_3d.cuh:16, src/cpu_3d.cpp:281-301).
//   tab : one sys_table per system: integer acceptance thresholds.
//
// Update order.  The reference CPU sweep (src/cpu_3d.cpp:94-105) visits, for
// offset 0 then 1, every site with (x+y)%2 == offset in z-major order and updates in
// place.  In 2D (and in-plane in 3D) neighbours of a site have the other colour
// (even L), so a half-sweep is data-parallel.  Along z, however, neighbours share
// the colour: site z reads the NEW value of z-1 and the OLD value of z+1; z = 0
// reads the old plane L-1 and z = L-1 the new plane 0.  The 3D kernel therefore
// gives each thread one (x,y) column of the current colour and walks z in order,
// carrying the new z-1 word and the new plane-0 word in registers: this is the
// reference's update order exactly, not a 3D checkerboard.
//
// Arithmetic is integer only: sat = J ^ s_i ^ s_j (bit set = satisfied bond), a
// bit-sliced full-adder tree gives the 3-bit satisfied count c per lane, the
// site's random word g is compared with the per-level thresholds, and a mux tree
// over c picks the flip mask.  One random word per site update is shared by the 64
// lanes, as in the reference (src/cpu_3d.cpp:130).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "sa/rng.hpp"

namespace sa {

enum { KIND_2P = 0, KIND_2D = 1, KIND_3D = 2 };

// Acceptance thresholds of one system.  Table 0/1: bulk sites with spin bit 0/1;
// table 2/3: open-x border sites (2p only).  Level c accepts iff g < thr[t][c]
// or bit c of always[t] is set.  base[t]: the table is compact -- levels below base[t]
// always accept, the others (at most four) have non-increasing thresholds -- so the
// accepted levels of a draw are 0 .. k-1 for one k; kNotCompact where it is not (a
// negative temperature, say).  Open-x border sites always count the missing bond, so
// their level 0 never occurs and counts as accepted.
struct sys_table {
  uint64_t thr[4][8];  // thr[t][7] is 0 (no such level)
  uint32_t always[4];
  uint32_t base[4];
};
constexpr uint32_t kNotCompact = 255;

struct sweep_args {
  uint64_t *s;
  const uint64_t *jx, *jy, *jz;
  const sys_table *tab;
  const uint64_t *words;  // replay: raw words of this sweep in visit order (N)
  uint64_t seed;          // counter mode key
  uint64_t sweep;         // counter mode: sweeps done since seeding
  int64_t N;
  int L;
  int nsys;
};

// ---------------------------------------------------------------- bit-sliced logic
// gfx950's v_bitop3_b32 evaluates any 3-input bitwise function in one VALU
// instruction; the 8-bit truth table of f is f(0xF0, 0xCC, 0xAA) for operands
// (a, b, c).  64-bit words are handled as two 32-bit halves.
constexpr int B3_XOR3 = 0x96;  // a ^ b ^ c
constexpr int B3_MAJ3 = 0xE8;  // majority(a, b, c)
constexpr int B3_MUX = 0xCA;   // a ? b : c, per bit
constexpr int B3_FLIP = 0x65;  // c ^ (~a | b): spin c flipped where ~a | b

template <int IMM>
__device__ __forceinline__ uint32_t b3(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, IMM);
}
template <int IMM>
__device__ __forceinline__ uint64_t b3(uint64_t a, uint64_t b, uint64_t c) {
  const uint32_t lo = __builtin_amdgcn_bitop3_b32((uint32_t)a, (uint32_t)b, (uint32_t)c, IMM);
  const uint32_t hi = __builtin_amdgcn_bitop3_b32((uint32_t)(a >> 32), (uint32_t)(b >> 32), (uint32_t)(c >> 32), IMM);
  return ((uint64_t)hi << 32) | lo;
}

struct count3 {
  uint64_t b0, b1, b2;
};

__device__ __forceinline__ uint64_t xor3(uint64_t a, uint64_t b, uint64_t c) { return b3<B3_XOR3>(a, b, c); }
__device__ __forceinline__ uint64_t maj3(uint64_t a, uint64_t b, uint64_t c) { return b3<B3_MAJ3>(a, b, c); }

// number of set bits among six words, per lane (0..6): two full adders and a
// third on the carries
__device__ __forceinline__ count3 count6(uint64_t a, uint64_t b, uint64_t c, uint64_t d, uint64_t e,
                                         uint64_t f) {
  const uint64_t s1 = xor3(a, b, c), k1 = maj3(a, b, c);
  const uint64_t s2 = xor3(d, e, f), k2 = maj3(d, e, f);
  const uint64_t k3 = s1 & s2;
  return count3{s1 ^ s2, xor3(k1, k2, k3), maj3(k1, k2, k3)};
}

// ... among four words (0..4)
__device__ __forceinline__ count3 count4(uint64_t a, uint64_t b, uint64_t c, uint64_t d) {
  const uint64_t s1 = xor3(a, b, c), k1 = maj3(a, b, c);
  const uint64_t k2 = s1 & d;
  return count3{s1 ^ d, k1 ^ k2, k1 & k2};
}

__device__ __forceinline__ uint64_t sel(uint64_t m, uint64_t a, uint64_t b) {  // m ? a : b, per bit
  return b3<B3_MUX>(m, a, b);
}

__device__ __forceinline__ uint64_t lvl(bool acc) { return acc ? ~0ULL : 0ULL; }

// per-level accept masks of one table for draw g (levels 0..7)
__device__ __forceinline__ void level_masks(const sys_table &t, int tb, uint64_t g, uint64_t a[8], int nlev) {
#pragma unroll
  for (int c = 0; c < 8; ++c)
    a[c] = (c < nlev) ? lvl((g < t.thr[tb][c]) || ((t.always[tb] >> c) & 1u)) : 0ULL;
}

// lane-wise a[c] with c given bit-sliced
__device__ __forceinline__ uint64_t mux8(const count3 &c, const uint64_t a[8]) {
  const uint64_t m0 = sel(c.b0, a[1], a[0]), m1 = sel(c.b0, a[3], a[2]);
  const uint64_t m2 = sel(c.b0, a[5], a[4]), m3 = sel(c.b0, a[7], a[6]);
  const uint64_t n0 = sel(c.b1, m1, m0), n1 = sel(c.b1, m3, m2);
  return sel(c.b2, n1, n0);
}

// New spin word of a site: general tables (any T, any h).
__device__ __forceinline__ uint64_t update_general(const sys_table &t, int tb0, uint64_t g, const count3 &c,
                                                   uint64_t si, int nlev) {
  uint64_t a[8];
  level_masks(t, tb0, g, a, nlev);
  const uint64_t f0 = mux8(c, a);
  level_masks(t, tb0 + 1, g, a, nlev);
  const uint64_t f1 = mux8(c, a);
  return si ^ sel(si, f1, f0);
}

// New spin word when both spin tables are equal and every level c <= nb/2 always
// accepts (h = 0, T > 0): only the levels above nb/2 need a comparison.  The
// accept decisions are per site, so they are built once as 32-bit masks and
// applied to both halves of the word.
//   3D (levels 4,5,6 thresholded): flip = ~c2 | (c1 ? a6 : (c0 ? a5 : a4))
//   2D (levels 3,4):               flip = c2 ? a4 : ((c1 & c0) ? a3 : ~0)
__device__ __forceinline__ uint64_t update_fast3t(uint64_t t4, uint64_t t5, uint64_t t6, uint64_t g, const count3 &c,
                                                  uint64_t si) {
  const uint32_t a4 = (g < t4) ? ~0u : 0u, a5 = (g < t5) ? ~0u : 0u;
  const uint32_t a6 = (g < t6) ? ~0u : 0u;
  const uint32_t vlo = b3<B3_MUX>((uint32_t)c.b1, a6, b3<B3_MUX>((uint32_t)c.b0, a5, a4));
  const uint32_t vhi = b3<B3_MUX>((uint32_t)(c.b1 >> 32), a6, b3<B3_MUX>((uint32_t)(c.b0 >> 32), a5, a4));
  const uint32_t lo = b3<B3_FLIP>((uint32_t)c.b2, vlo, (uint32_t)si);
  const uint32_t hi = b3<B3_FLIP>((uint32_t)(c.b2 >> 32), vhi, (uint32_t)(si >> 32));
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t update_fast3(const sys_table &t, uint64_t g, const count3 &c, uint64_t si) {
  return update_fast3t(t.thr[0][4], t.thr[0][5], t.thr[0][6], g, c, si);
}
__device__ __forceinline__ uint64_t update_fast2(const sys_table &t, uint64_t g, const count3 &c, uint64_t si) {
  const uint64_t a3 = lvl(g < t.thr[0][3]), a4 = lvl(g < t.thr[0][4]);
  return si ^ sel(c.b2, a4, ~(c.b1 & c.b0) | a3);
}

// ---------------------------------------------------------------- buffer access
// Raw buffer loads/stores: a 128-bit resource (base, size) in scalar registers, a
// per-thread 32-bit byte offset that stays fixed for the whole z-walk, and the
// plane offset as a wave-uniform scalar -- no per-load 64-bit address arithmetic.
typedef unsigned int sa_v2u32 __attribute__((ext_vector_type(2)));
typedef unsigned int sa_v4u32 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t buf_t;

// A buffer access whose per-thread offset is at or beyond the resource size is
// discarded by the hardware range check: loads return 0 and stores write nothing.
// Lanes and planes with nothing to load or store use this offset, so every load
// and store instruction of the z-walk is issued unconditionally and the compiler
// can count the outstanding loads exactly (no drain of the prefetch).
constexpr uint32_t kOutOfRange = 0x80000000u;

__device__ __forceinline__ buf_t make_buf(const void *p, uint32_t bytes) {
  // dword 3 = 0x00020000: raw (untyped) dword access on gfx9-family GPUs
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint64_t bld(buf_t b, uint32_t voff, uint32_t soff) {
  const sa_v2u32 v = __builtin_amdgcn_raw_buffer_load_b64(b, (int)voff, (int)soff, 0);
  return ((uint64_t)v.y << 32) | v.x;
}
// Cache policy of a load / store (gfx950: bit 1 = "nt", non-temporal).  The fused
// sweep reads each old spin pair once and writes each new pair once per sweep, and
// a ladder's spins are far larger than the last-level cache, so that traffic is
// marked non-temporal; couplings (read by every system block) and the halo rows
// (read by two bands) keep the default policy.  Measured on the 3D L=128, 32-system
// sweep: 309 -> 283 us per launch.
constexpr int kCpolNT = 2;
#ifndef SA_FUSED_PAIR_CPOL
#define SA_FUSED_PAIR_CPOL kCpolNT
#endif
template <int CPOL = 0>
__device__ __forceinline__ void bld2(buf_t b, uint32_t voff, uint32_t soff, uint64_t &a, uint64_t &c) {
  const sa_v4u32 v = __builtin_amdgcn_raw_buffer_load_b128(b, (int)voff, (int)soff, CPOL);
  a = ((uint64_t)v.y << 32) | v.x;
  c = ((uint64_t)v.w << 32) | v.z;
}
template <int CPOL = 0>
__device__ __forceinline__ void bst2(buf_t b, uint32_t voff, uint32_t soff, uint64_t a, uint64_t c) {
  sa_v4u32 v;
  v.x = (uint32_t)a;
  v.y = (uint32_t)(a >> 32);
  v.z = (uint32_t)c;
  v.w = (uint32_t)(c >> 32);
  __builtin_amdgcn_raw_buffer_store_b128(v, b, (int)voff, (int)soff, CPOL);
}

// ---------------------------------------------------------------- 3D half-sweep
// Thread = one column (x, y) of colour `color` and MB systems; grid.y = system
// block (so thresholds are wave-uniform and live in scalar registers).
//
// Software pipeline: nothing a step loads depends on the step before it (the
// in-plane neighbours have the other colour and do not change during the half;
// the column's own next word is still old), so the loads of step z+1 are issued
// before the arithmetic and the store of step z and overlap its latency.
template <int MB>
struct plane_loads {
  uint64_t jw, je, jn, js, jd;  // couplings: -x, +x, -y, +y, +z bonds
  uint64_t w[MB], e[MB], n[MB], s[MB], d[MB];
};

// column k (0 <= k < L*L/2) of colour `color`, systems sys0 .. sys0+MB-1
// DEEP: plane loads issued two planes ahead instead of one (more registers; pays
// where few long column walks set the pace, as in the batched engine)
template <bool COUNTER, bool FAST, int MB, bool DEEP = false>
__device__ __forceinline__ void half3d_column(const sweep_args &p, int color, int k, int sys0) {
  const int L = p.L;
  const int half = L >> 1;
  const int y = k / half;
  const int x = 2 * (k - y * half) + ((y + color) & 1);
  const int xm = x == 0 ? L - 1 : x - 1, xp = x == L - 1 ? 0 : x + 1;
  const int ym = y == 0 ? L - 1 : y - 1, yp = y == L - 1 ? 0 : y + 1;
  const int64_t L2 = (int64_t)L * L;
  const int c0 = x + L * y;               // in-plane offsets
  const int cw = xm + L * y, ce = xp + L * y, cn = x + L * ym, cs = x + L * yp;
  const int64_t N = p.N;
  const int64_t rank0 = (int64_t)color * (N >> 1) + k;  // visit rank of (x,y,0)
  const int64_t rstep = L2 >> 1;

  uint64_t *sp[MB];
  uint64_t up[MB], own[MB], first[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    sp[m] = p.s + (int64_t)(sys0 + m) * N;
    up[m] = sp[m][c0 + (L - 1) * L2];     // old plane L-1
    own[m] = sp[m][c0];
    first[m] = 0;
  }
  // loads of plane z (the +z neighbour of plane L-1 is the new plane 0: not loaded)
  auto load = [&](int z, plane_loads<MB> &q) {
    const int64_t P = z * L2;
    const int64_t Pd = (z == L - 1) ? 0 : P + L2;
    q.jw = p.jx[P + c0];
    q.je = p.jx[P + ce];
    q.jn = p.jy[P + c0];
    q.js = p.jy[P + cs];
    q.jd = p.jz[Pd + c0];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const uint64_t *s = sp[m];
      q.w[m] = s[P + cw];
      q.e[m] = s[P + ce];
      q.n[m] = s[P + cn];
      q.s[m] = s[P + cs];
      q.d[m] = (z == L - 1) ? 0 : s[Pd + c0];
    }
  };
  uint64_t jz_up = p.jz[c0];
  u32x4 blk{0, 0, 0, 0};
  // DEEP: plane z's loads are issued two planes ahead, three buffers rotating
  // through the z loop unrolled by 3; otherwise one plane ahead.
  auto plane = [&](int z, const plane_loads<MB> &cur, plane_loads<MB> &far, int ahead) {
    if (z + ahead < L) load(z + ahead, far);
    uint64_t g;
    if (COUNTER) {
      if ((z & 1) == 0) blk = counter_block((uint32_t)(c0 + z * L2), p.seed, p.sweep);
      g = counter_half(blk, z & 1);
    } else {
      g = p.words[rank0 + z * rstep];
    }
    const int64_t P = z * L2;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const uint64_t si = own[m];
      const uint64_t down = (z == L - 1) ? first[m] : cur.d[m];
      const count3 c = count6(xor3(cur.jw, si, cur.w[m]), xor3(cur.je, si, cur.e[m]), xor3(cur.jn, si, cur.n[m]),
                              xor3(cur.js, si, cur.s[m]), xor3(jz_up, si, up[m]), xor3(cur.jd, si, down));
      const sys_table &t = p.tab[sys0 + m];
      const uint64_t sn = FAST ? update_fast3(t, g, c, si) : update_general(t, 0, g, c, si, 7);
      sp[m][P + c0] = sn;
      up[m] = sn;
      if (z == 0) first[m] = sn;
      own[m] = down;
    }
    jz_up = cur.jd;
  };
  if constexpr (DEEP) {
    plane_loads<MB> b0, b1, b2;
    load(0, b0);
    if (1 < L) load(1, b1);
    for (int z = 0; z < L; z += 3) {
      plane(z, b0, b2, 2);
      if (z + 1 < L) plane(z + 1, b1, b0, 2);
      if (z + 2 < L) plane(z + 2, b2, b1, 2);
    }
  } else {
    plane_loads<MB> cur, nxt;
    load(0, cur);
    for (int z = 0; z < L; ++z) {
      plane(z, cur, nxt, 1);
      cur = nxt;
    }
  }
}

template <bool COUNTER, bool FAST, int MB>
__global__ void __launch_bounds__(256) k_sweep3d_half(sweep_args p, int color) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= p.L * (p.L >> 1)) return;
  half3d_column<COUNTER, FAST, MB>(p, color, k, blockIdx.y * MB);
}

// ---------------------------------------------------------------- 3D fused sweep
// One launch per sweep.  A workgroup owns a band of TH full rows (y0 .. y0+TH-1)
// of MB systems and walks z once; at every plane it performs the offset-0 half
// (colour 0) and then the offset-1 half (colour 1):
//   * colour-0 site at plane z needs old colour-1 in-plane neighbours, the new
//     colour-0 word at z-1 and the old one at z+1 -- exactly what the reference's
//     first half-sweep sees there, since that half never touches colour 1 and walks
//     z upwards (src/cpu_3d.cpp:94-105);
//   * colour-1 site at plane z needs the NEW colour-0 in-plane neighbours of the
//     same plane, the new colour-1 word at z-1 and the old one at z+1.
// The colour-0 updates of the rows just outside the band (y0-1, y0+TH) are
// recomputed by the workgroup (identical to the neighbour's), so no workgroup
// waits for another.  Spins are read from one array and written to another
// (ping-pong per sweep), so every "old" value a workgroup reads is untouched by
// any other workgroup during the sweep.
//
// Threads: (TH+2) rows x L/2 site pairs (2k, 2k+1); row 0 and row TH+1 are the
// halo rows.  LDS holds, per plane buffer, row and system, the colour-0 and the
// colour-1 word of every pair: c0[k], c1[k].  In a row of parity P the colour-0
// site of pair k is x0 = 2k+P and the colour-1 site x1 = 2k+1-P, so
//   colour-0 x-neighbours: c1[k], c1[k + (P ? 1 : -1)]   y-neighbours: c1[k] of rows r-1, r+1
//   colour-1 x-neighbours: c0[k], c0[k + (P ? -1 : 1)]   y-neighbours: c0[k] of rows r-1, r+1
// One barrier per plane: iteration z updates colour 1 of plane z and colour 0 of
// plane z+1 (which reads only old colour-1 words of plane z+1 and the column's own
// colour-0 chain) and stores the old words of plane z+2; three LDS plane buffers
// rotate.  A thread's row parity is fixed, so the z-walk is instantiated per
// parity when a row spans whole waves (L/2 a multiple of 64), where the choice is
// wave-uniform; smaller lattices keep the parity as a run-time value.
template <int MB>
struct fused_loads {
  uint64_t na[MB], nb[MB];  // own pair at plane z+1 (old)
  uint64_t ring2[MB];       // halo rows: colour-1 word one row further out (old)
  uint64_t jxa, jxb, jxn;   // jx of 2k, 2k+1, 2k+2
  uint64_t jya, jyb;        // jy of the pair (bond to y-1)
  uint64_t jsa, jsb;        // jy of the pair in row y+1 (bond to y+1)
  uint64_t jda, jdb;        // jz of the pair at plane z+1 (bond to z+1)
  uint64_t g0, g1;          // replay words of the colour-0 / colour-1 site
};

template <bool COUNTER, bool FAST, int MB, int TH>
struct fused_ctx {
  const sweep_args &p;
  uint64_t *lds;
  int L, PR, r, rn, rs, k, kn, kp, y, row, rowS, yr2, sys0;
  uint32_t t_rk, t_rkp, t_rkn, t_rnk, t_rsk;  // per-thread LDS byte offsets (see at())
  uint64_t t4[MB], t5[MB], t6[MB];  // FAST: the thresholded levels of each system's table
  bool halo;
  int64_t L2, N, rank0;
  int par;  // row parity (the template argument P is -1 when it is only known at run time)
  buf_t sin[MB], sout[MB], bjx, bjy, bjz, bw;
  uint32_t vpair, vpairS, vnext, vring, vrank, vrank1, vstore;  // per-thread byte offsets
  uint32_t plane_bytes;                          // L*L*8

  // LDS word of (plane buffer, system m, colour c) at a thread position.  The
  // element index (((buf*(TH+2) + row)*MB + m)*2 + c)*PR + col splits into a
  // wave-uniform slab offset (buf, m, c) and a per-thread offset (row, col) that is
  // fixed for the walk (t_rk .. t_rsk), so an access costs one add.
  __device__ __forceinline__ uint32_t slab(int buf, int m, int c) const {
    return (uint32_t)((buf * (TH + 2) * MB * 2 + m * 2 + c) * PR) * 8u;
  }
  __device__ __forceinline__ uint64_t &at(uint32_t slab_off, uint32_t toff) const {
    return *reinterpret_cast<uint64_t *>(reinterpret_cast<char *>(lds) + slab_off + toff);
  }
  // WROW: a row is one whole wave (L/2 == 64); jx of pair k+1 then comes from the
  // next lane at use time instead of a load
  template <bool WROW>
  __device__ __forceinline__ void load(int z, fused_loads<MB> &q) const {
    const bool top = z == L - 1;
    const uint32_t P = (uint32_t)z * plane_bytes;
    const uint32_t Pd = top ? 0u : P + plane_bytes;
    const uint32_t vn = top ? kOutOfRange : vpair;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      bld2<SA_FUSED_PAIR_CPOL>(sin[m], vn, Pd, q.na[m], q.nb[m]);
      q.ring2[m] = bld(sin[m], vring, P);
    }
    bld2(bjx, vpair, P, q.jxa, q.jxb);
    if (!WROW) q.jxn = bld(bjx, vnext, P);
    bld2(bjy, vpair, P, q.jya, q.jyb);
    bld2(bjy, vpairS, P, q.jsa, q.jsb);
    bld2(bjz, vpair, Pd, q.jda, q.jdb);
    if (!COUNTER) {
      const uint32_t half_plane = (uint32_t)z * (plane_bytes >> 1);
      q.g0 = bld(bw, vrank, half_plane);
      q.g1 = bld(bw, vrank1, half_plane + (uint32_t)(N >> 1) * 8u);
    }
  }

  // What the colour-1 update of a plane needs, captured right after the colour-0
  // update of the same plane.
  struct bstate {
    uint64_t jw, je, jn, js, jd, g;
    uint64_t si[MB], down[MB], n0[MB];
  };

  // in-plane neighbour words of the thread's site of one colour, per system
  struct nbrs {
    uint64_t w[MB], e[MB], n[MB], s[MB];
  };
  // Both phases' LDS reads are issued together at the top of an iteration (they
  // read different plane buffers than the iteration writes), so a wave waits for
  // LDS once per plane.  Rows rn/rs are r-1/r+1 clamped to the band: the halo
  // rows take ring2 instead, or do not use the values (phase B).
  template <int PT>
  __device__ __forceinline__ void read_a(int q, const fused_loads<MB> &ld, nbrs &v) const {
    const int P = PT >= 0 ? PT : par;
    const int buf = q % 3;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const uint32_t sl = slab(buf, m, 1);
      v.w[m] = at(sl, P ? t_rk : t_rkp);
      v.e[m] = at(sl, P ? t_rkn : t_rk);
      const uint64_t nn = at(sl, t_rnk), ss = at(sl, t_rsk);
      v.n[m] = (r == 0) ? ld.ring2[m] : nn;
      v.s[m] = (r == TH + 1) ? ld.ring2[m] : ss;
    }
  }
  template <int PT>
  __device__ __forceinline__ void read_b(int q, nbrs &v) const {
    const int P = PT >= 0 ? PT : par;
    const int buf = q % 3;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const uint32_t sl = slab(buf, m, 0);
      v.w[m] = at(sl, P ? t_rkp : t_rk);
      v.e[m] = at(sl, P ? t_rk : t_rkn);
      v.n[m] = at(sl, t_rnk);
      v.s[m] = at(sl, t_rsk);
    }
  }

  // colour-0 update of plane q (all rows, halo included).  q_loads holds the loads
  // of plane q, pair[] the old pair at plane q, v the colour-1 neighbours.  Writes
  // the new colour-0 words into LDS buffer q%3 and fills bs for the colour-1 update
  // of plane q.
  template <int PT>
  __device__ __forceinline__ void phase_a(int q, const fused_loads<MB> &ld, const nbrs &v, const uint64_t *pa,
                                          const uint64_t *pb, uint64_t g0, uint64_t g1, uint64_t *up0,
                                          uint64_t *first0, const uint64_t *first1, uint64_t &ju0, bstate &bs) const {
    const int P = PT >= 0 ? PT : par;
    const int buf = q % 3;
    const bool last = q == L - 1;
    // jx of 2k+2: the next pair's jxa (lane k+1 of the same row) when a row is a wave
    const uint64_t jxn = PT >= 0 ? __shfl(ld.jxa, (int)((threadIdx.x + 1) & 63)) : ld.jxn;
    const uint64_t j0w = P ? ld.jxb : ld.jxa, j0e = P ? jxn : ld.jxb;
    const uint64_t j0n = P ? ld.jyb : ld.jya, j0s = P ? ld.jsb : ld.jsa;
    const uint64_t j0d = P ? ld.jdb : ld.jda;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const uint64_t si = P ? pb[m] : pa[m];
      const uint64_t w = v.w[m], e = v.e[m], nn = v.n[m], ss = v.s[m];
      const uint64_t down = last ? first0[m] : (P ? ld.nb[m] : ld.na[m]);
      const count3 c = count6(xor3(j0w, si, w), xor3(j0e, si, e), xor3(j0n, si, nn), xor3(j0s, si, ss),
                              xor3(ju0, si, up0[m]), xor3(j0d, si, down));
      const uint64_t n0 =
          FAST ? update_fast3t(t4[m], t5[m], t6[m], g0, c, si) : update_general(p.tab[sys0 + m], 0, g0, c, si, 7);
      at(slab(buf, m, 0), t_rk) = n0;
      up0[m] = n0;
      if (q == 0) first0[m] = n0;
      bs.si[m] = P ? pa[m] : pb[m];
      bs.down[m] = last ? first1[m] : (P ? ld.na[m] : ld.nb[m]);
      bs.n0[m] = n0;
    }
    ju0 = j0d;
    bs.jw = P ? ld.jxa : ld.jxb;
    bs.je = P ? ld.jxb : jxn;
    bs.jn = P ? ld.jya : ld.jyb;
    bs.js = P ? ld.jsa : ld.jsb;
    bs.jd = P ? ld.jda : ld.jdb;
    bs.g = g1;
  }

  // colour-1 update of plane q (band rows): reads the new colour-0 words of plane q
  // from LDS buffer q%3; oa/ob = the pair's new words (x = 2k, 2k+1).
  template <int PT>
  __device__ __forceinline__ void phase_b(int q, const nbrs &v, const bstate &bs, uint64_t *up1, uint64_t *first1,
                                          uint64_t &ju1, uint64_t *oa, uint64_t *ob) const {
    const int P = PT >= 0 ? PT : par;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const uint64_t si = bs.si[m];
      const uint64_t w = v.w[m], e = v.e[m], nn = v.n[m], ss = v.s[m];
      const count3 c = count6(xor3(bs.jw, si, w), xor3(bs.je, si, e), xor3(bs.jn, si, nn), xor3(bs.js, si, ss),
                              xor3(ju1, si, up1[m]), xor3(bs.jd, si, bs.down[m]));
      const uint64_t n1 = FAST ? update_fast3t(t4[m], t5[m], t6[m], bs.g, c, si)
                               : update_general(p.tab[sys0 + m], 0, bs.g, c, si, 7);
      up1[m] = n1;
      if (q == 0) first1[m] = n1;
      oa[m] = P ? n1 : bs.n0[m];
      ob[m] = P ? bs.n0[m] : n1;
    }
    ju1 = bs.jd;
  }

  // old colour-1 word of plane q into LDS buffer q%3.  The old colour-0 word is not
  // stored: nothing reads it from LDS (phase A of plane q writes the new one into the
  // same slot before any phase B reads the slot).
  template <int PT>
  __device__ __forceinline__ void put_old(int q, const uint64_t *pa, const uint64_t *pb) const {
    const int P = PT >= 0 ? PT : par;
    const int buf = q % 3;
#pragma unroll
    for (int m = 0; m < MB; ++m) at(slab(buf, m, 1), t_rk) = P ? pa[m] : pb[m];
  }

  // random words of the colour-0 / colour-1 site at plane q
  __device__ __forceinline__ void words(int q, const fused_loads<MB> &ld, int x0, int x1, u32x4 &blk0, u32x4 &blk1,
                                        uint64_t &g0, uint64_t &g1) const {
    if (COUNTER) {
      if ((q & 1) == 0) {
        blk0 = counter_block((uint32_t)(x0 + row + q * L2), p.seed, p.sweep);
        if (!halo) blk1 = counter_block((uint32_t)(x1 + row + q * L2), p.seed, p.sweep);
      }
      g0 = counter_half(blk0, q & 1);
      g1 = counter_half(blk1, q & 1);
    } else {
      g0 = ld.g0;
      g1 = ld.g1;
    }
  }

  // One pass over z.  Iteration z: colour-1 update of plane z, colour-0 update of
  // plane z+1, old words of plane z+2 into LDS, one barrier.  Phase A(z+1) may run
  // before phase B(z) finishes elsewhere: it reads only old colour-1 words of plane
  // z+1 and the column's own colour-0 chain.  Three LDS plane buffers: z (read by
  // phase B), z+1 (phase A), z+2 (being filled).
  template <int PT>
  __device__ __forceinline__ void walk() const {
    const int P = PT >= 0 ? PT : par;
    const int x0 = 2 * k + P, x1 = 2 * k + 1 - P;
    uint64_t pa[MB], pb[MB], up0[MB], up1[MB], first0[MB], first1[MB];
    const uint32_t top = (uint32_t)(L - 1) * plane_bytes;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      bld2(sin[m], vpair, 0u, pa[m], pb[m]);
      uint64_t ta, tb;
      bld2(sin[m], vpair, top, ta, tb);  // old plane L-1
      up0[m] = P ? tb : ta;
      up1[m] = P ? ta : tb;
      first0[m] = first1[m] = 0;
    }
    uint64_t ja, jb;
    bld2(bjz, vpair, 0u, ja, jb);  // -z bonds at plane 0
    uint64_t ju0 = P ? jb : ja, ju1 = P ? ja : jb;
    u32x4 blk0{0, 0, 0, 0}, blk1{0, 0, 0, 0};
    fused_loads<MB> A, B;  // loads of planes z+1 / z+2, used alternately
    bstate bs;
    // prologue: old planes 0 and 1 into LDS, colour-0 update of plane 0
    load<PT >= 0>(0, A);
    load<PT >= 0>(1, B);
    put_old<PT>(0, pa, pb);
    put_old<PT>(1, A.na, A.nb);
    __syncthreads();
    {
      uint64_t g0, g1;
      nbrs va;
      read_a<PT>(0, A, va);
      words(0, A, x0, x1, blk0, blk1, g0, g1);
      phase_a<PT>(0, A, va, pa, pb, g0, g1, up0, first0, first1, ju0, bs);
    }
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      pa[m] = A.na[m];  // old pair at plane 1
      pb[m] = A.nb[m];
    }
    __syncthreads();
    // iteration z: near = loads of plane z+1, far = loads of plane z+2 (prefetched)
    auto iteration = [&](int z, fused_loads<MB> &near, fused_loads<MB> &far) {
      load<PT >= 0>(z + 2 < L ? z + 2 : L - 1, far);  // the last two loads are not used
      nbrs vb;
      read_b<PT>(z, vb);
      {
        uint64_t oa[MB], ob[MB];
        if (!halo) {
          phase_b<PT>(z, vb, bs, up1, first1, ju1, oa, ob);
        } else {
#pragma unroll
          for (int m = 0; m < MB; ++m) oa[m] = ob[m] = 0;
        }
#pragma unroll
        for (int m = 0; m < MB; ++m) bst2<SA_FUSED_PAIR_CPOL>(sout[m], vstore, (uint32_t)z * plane_bytes, oa[m], ob[m]);
      }
      if (z + 1 < L) {
        uint64_t g0, g1;
        nbrs va;
        read_a<PT>(z + 1, near, va);
        words(z + 1, near, x0, x1, blk0, blk1, g0, g1);
        phase_a<PT>(z + 1, near, va, pa, pb, g0, g1, up0, first0, first1, ju0, bs);
        if (z + 2 < L) put_old<PT>(z + 2, near.na, near.nb);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          pa[m] = near.na[m];  // old pair at plane z+2
          pb[m] = near.nb[m];
        }
      }
      __syncthreads();
    };
    for (int z = 0; z < L; z += 2) {  // L is even
      iteration(z, B, A);
      iteration(z + 1, A, B);
    }
  }
};

// One workgroup's band `tile` of system block `sb` (systems sb*MB .. sb*MB+MB-1):
// the whole z-walk.  blockDim.x must be (TH+2)*L/2 and the dynamic LDS
// 3*(TH+2)*MB*2*(L/2)*8 bytes.
// WALK: 1 = rows are whole waves (L/2 a multiple of 64), 0 = they are not, 2 = decide
// at run time (both walks compiled in).
template <bool COUNTER, bool FAST, int MB, int TH, int WALK = 2>
__device__ __forceinline__ void fused_band(const sweep_args &p, uint64_t *__restrict__ s_out, int sb, int tile,
                                           uint64_t *lds) {
  const int L = p.L, PR = L >> 1;
  fused_ctx<COUNTER, FAST, MB, TH> c{p, lds};
  c.L = L;
  c.PR = PR;
  c.r = threadIdx.x / PR;
  c.k = threadIdx.x - c.r * PR;
  c.kn = c.k == PR - 1 ? 0 : c.k + 1;
  c.kp = c.k == 0 ? PR - 1 : c.k - 1;
  c.halo = (c.r == 0) || (c.r == TH + 1);
  c.rn = c.r == 0 ? 0 : c.r - 1;
  c.rs = c.r == TH + 1 ? TH + 1 : c.r + 1;
  {
    const uint32_t rowst = (uint32_t)(MB * 2 * PR);  // elements per LDS row (all systems, both colours)
    c.t_rk = ((uint32_t)c.r * rowst + (uint32_t)c.k) * 8u;
    c.t_rkp = ((uint32_t)c.r * rowst + (uint32_t)c.kp) * 8u;
    c.t_rkn = ((uint32_t)c.r * rowst + (uint32_t)c.kn) * 8u;
    c.t_rnk = ((uint32_t)c.rn * rowst + (uint32_t)c.k) * 8u;
    c.t_rsk = ((uint32_t)c.rs * rowst + (uint32_t)c.k) * 8u;
  }
  c.y = (tile * TH - 1 + c.r + L) % L;
  const int ym = c.y == 0 ? L - 1 : c.y - 1, yp = c.y == L - 1 ? 0 : c.y + 1;
  c.row = c.y * L;
  c.rowS = yp * L;
  c.yr2 = (c.r == 0) ? ym : yp;  // halo rows: the row beyond the halo
  c.sys0 = sb * MB;
#pragma unroll
  for (int m = 0; m < MB; ++m) {  // loaded once for the whole walk
    const sys_table &t = p.tab[c.sys0 + m];
    c.t4[m] = t.thr[0][4];
    c.t5[m] = t.thr[0][5];
    c.t6[m] = t.thr[0][6];
  }
  c.L2 = (int64_t)L * L;
  c.N = p.N;
  c.rank0 = (int64_t)c.y * PR + c.k;  // visit rank inside a plane half
  const uint32_t bytes = (uint32_t)(c.N * 8);
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    c.sin[m] = make_buf(p.s + (int64_t)(c.sys0 + m) * c.N, bytes);
    c.sout[m] = make_buf(s_out + (int64_t)(c.sys0 + m) * c.N, bytes);
  }
  c.bjx = make_buf(p.jx, bytes);
  c.bjy = make_buf(p.jy, bytes);
  c.bjz = make_buf(p.jz, bytes);
  c.bw = make_buf(p.words, COUNTER ? 0u : bytes);
  c.plane_bytes = (uint32_t)(c.L2 * 8);
  c.vpair = (uint32_t)(c.row + 2 * c.k) * 8u;
  c.vpairS = (uint32_t)(c.rowS + 2 * c.k) * 8u;
  c.vnext = (uint32_t)(c.row + 2 * c.kn) * 8u;
  c.vring = c.halo ? (uint32_t)(c.yr2 * L + 2 * c.k + (c.y & 1)) * 8u : kOutOfRange;
  c.vrank = (uint32_t)c.rank0 * 8u;
  c.vrank1 = c.halo ? kOutOfRange : c.vrank;  // halo rows do not update colour 1
  c.vstore = c.halo ? kOutOfRange : c.vpair;  // nor store anything
  c.par = c.y & 1;
  // The walk contains barriers, so a parity-specialised walk may only be chosen
  // per wave: when a row is a whole number of waves (L/2 a multiple of 64) every
  // wave has one parity; otherwise the parity stays a run-time value.
  if (WALK == 1 || (WALK == 2 && (PR & 63) == 0)) {
    if (c.par) c.template walk<1>(); else c.template walk<0>();
  } else {
    c.template walk<-1>();
  }
}

// Compiled once per walk (WALK 0 or 1, see fused_band): one kernel holding both
// walks allocates registers for both and runs slower.
template <bool COUNTER, bool FAST, int MB, int TH, int WALK>
__global__ void __launch_bounds__(640) k_sweep3d_fused(sweep_args p, uint64_t *__restrict__ s_out, int xcd_map) {
  extern __shared__ uint64_t lds[];
  const int ntile = p.L / TH;
  // workgroup -> (system block, band).  Workgroups are dispatched round-robin over
  // the 8 XCDs (L2 is per XCD).  xcd_map = 0: b = sb*ntile + band, so with ntile a
  // multiple of 8 every system block of a band runs on one XCD and shares its
  // couplings in L2.  xcd_map = 1: XCD b%8 gets ntile/8 adjacent bands of every
  // system block, so the halo rows between those bands are L2 hits too.
  // xcd_map = 2: XCD b%8 gets every band of nsb/8 whole system blocks, so every halo
  // row a band reads is read by its neighbour band on the same XCD (the couplings
  // are then read once per XCD).
  const int b = blockIdx.x;
  int sb, tile;
  if (xcd_map == 2) {
    const int per = (p.nsys / MB) >> 3, xcd = b & 7, q = b >> 3;
    sb = xcd * per + q / ntile;
    tile = q % ntile;
  } else if (xcd_map) {
    const int per = ntile >> 3, xcd = b & 7, q = b >> 3;
    tile = xcd * per + q % per;
    sb = q / per;
  } else {
    sb = b / ntile;
    tile = b - sb * ntile;
  }
  fused_band<COUNTER, FAST, MB, TH, WALK>(p, s_out, sb, tile, lds);
}

// ---------------------------------------------------------------- 3D half-sweep, z in parallel
// For a lattice too small to fill the GPU with column walks (one system offers L*L/2
// columns per half-sweep), each column is cut into G segments of S = L/G planes, one
// thread per segment, the G threads of a column in one wave: a wave holds C = 64/G
// consecutive columns, lane = segment*C + column, so C neighbouring lanes read
// neighbouring columns of one plane.
// In a half-sweep the in-plane neighbours have the other colour and stay fixed, and
// the old +z word is fixed, so the new word of plane z is a per-lane function of the
// new word of plane z-1 only: one of the four maps of a bit, kept as the pair
// (f0, f1) = (result for a 0 below, result for a 1 below) -- two evaluations of the
// update with the -z neighbour all zeros and all ones, sharing the site's random
// word.  Plane 0 reads the old plane L-1, so its map is constant; plane L-1 reads the
// new plane 0 as its +z neighbour, which the segment-0 lane has computed first and
// passes on.  Maps compose as (F o G)(b) = G(b) ? F1 : F0 per bit; a scan over the
// G lanes gives every segment the new word below it, and each segment then applies
// its maps in order and stores.  The result is the reference's in-order z walk bit
// for bit (src/cpu_3d.cpp:94-105), with the same random word per site.  All loads of
// a wave complete before its scan, so no segment's store meets a read of another.
struct zmap {
  uint64_t f0, f1;
};
__device__ __forceinline__ zmap zcompose(const zmap &F, const zmap &G) {  // F o G
  return zmap{sel(G.f0, F.f1, F.f0), sel(G.f1, F.f1, F.f0)};
}
__device__ __forceinline__ uint64_t shfl_up64(uint64_t v, int d, int width) {
  const uint32_t lo = __shfl_up((uint32_t)v, d, width), hi = __shfl_up((uint32_t)(v >> 32), d, width);
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t shfl64(uint64_t v, int src) {
  const uint32_t lo = __shfl((uint32_t)v, src), hi = __shfl((uint32_t)(v >> 32), src);
  return ((uint64_t)hi << 32) | lo;
}

// segments per column for an even L: a power of two G <= 64 with L/G <= kZsegMax
// planes per segment and at least two planes; 0 when there is none.  Two planes per
// segment while a wave still holds two or more columns (G <= 32), else the fewest
// segments of at most 4 planes, else of at most 8.  Measured per sweep of one system:
// L=64 13.0 us with 2-plane segments, 13.9 with 4; L=32 7.9 / 9.6; L=128 63 with 4
// (32 segments, two columns per wave) against 94 with 2 (one column per wave).
constexpr int kZsegMax = 8;
__host__ __device__ __forceinline__ int zscan_groups(int L) {
  const int h = L / 2;
  if (L >= 4 && L % 2 == 0 && h <= 32 && (h & (h - 1)) == 0) return h;
  for (int G = 2; G <= 64; G *= 2)
    if (L % G == 0 && L / G <= 4 && L / G >= 2) return G;
  for (int G = 2; G <= 64; G *= 2)
    if (L % G == 0 && L / G <= kZsegMax && L / G >= 2) return G;
  return 0;
}

template <bool COUNTER, bool FAST, int S>
__device__ __forceinline__ void zscan_segment(const sweep_args &p, int color, int k, int g, int G, int sys, bool live) {
  const int L = p.L, half = L >> 1;
  const int y = k / half;
  const int x = 2 * (k - y * half) + ((y + color) & 1);
  const int xm = x == 0 ? L - 1 : x - 1, xp = x == L - 1 ? 0 : x + 1;
  const int ym = y == 0 ? L - 1 : y - 1, yp = y == L - 1 ? 0 : y + 1;
  const int64_t L2 = (int64_t)L * L, N = p.N;
  const int c0 = x + L * y, cw = xm + L * y, ce = xp + L * y, cn = x + L * ym, cs = x + L * yp;
  uint64_t *s = p.s + (int64_t)sys * N;
  const sys_table &t = p.tab[sys];
  const int z0 = g * S;
  const int lane = threadIdx.x & 63, C = 64 / G, base = lane % C;  // base: the column's segment-0 lane
  auto eval = [&](uint64_t g64, const uint64_t *q, uint64_t si, uint64_t bd, uint64_t bu) {
    const count3 cc = count6(q[0], q[1], q[2], q[3], bd, bu);
    return FAST ? update_fast3(t, g64, cc, si) : update_general(t, 0, g64, cc, si, 7);
  };
  // every load of the segment first (a dead lane reads column 0: valid addresses),
  // then the arithmetic: the planes' memory round trips overlap
  uint64_t si[S], nb[S][4], jb[S][4], ju[S], jd[S], dn[S], g64[S], q[S][4];
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const int z = z0 + j;
    const int64_t P = z * L2;
    si[j] = s[P + c0];
    nb[j][0] = s[P + cw];
    nb[j][1] = s[P + ce];
    nb[j][2] = s[P + cn];
    nb[j][3] = s[P + cs];
    jb[j][0] = p.jx[P + c0];
    jb[j][1] = p.jx[P + ce];
    jb[j][2] = p.jy[P + c0];
    jb[j][3] = p.jy[P + cs];
    ju[j] = p.jz[P + c0];
    jd[j] = p.jz[(z == L - 1 ? 0 : P + L2) + c0];
    dn[j] = s[(z == L - 1 ? 0 : P + L2) + c0];  // plane L-1: replaced by the new plane 0 below
    if (!COUNTER) g64[j] = p.words[(int64_t)color * (N >> 1) + k + z * (L2 >> 1)];
  }
  const uint64_t up0 = s[(L - 1) * L2 + c0];  // old plane L-1: plane 0's -z neighbour
  if (COUNTER) {
    u32x4 blk{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < S; ++j) {
      const int z = z0 + j;
      if (j == 0 || (z & 1) == 0) blk = counter_block((uint32_t)(c0 + (z & ~1) * L2), p.seed, p.sweep);
      g64[j] = counter_half(blk, z & 1);
    }
  }
  zmap F[S];
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const int z = z0 + j;
#pragma unroll
    for (int r = 0; r < 4; ++r) q[j][r] = xor3(jb[j][r], si[j], nb[j][r]);
    const uint64_t bu0 = z == 0 ? xor3(ju[j], si[j], up0) : (ju[j] ^ si[j]);  // -z bond word, 0 below
    const uint64_t bd = xor3(jd[j], si[j], dn[j]);
    F[j].f0 = eval(g64[j], q[j], si[j], bd, bu0);
    F[j].f1 = z == 0 ? F[j].f0 : eval(g64[j], q[j], si[j], bd, ~bu0);  // plane 0: a constant map
  }
  // the new plane 0 (segment 0's constant map) to every lane of the column
  const uint64_t new0 = shfl64(F[0].f0, base);
  if (z0 + S == L) {  // plane L-1: its +z neighbour is the new plane 0
    constexpr int j = S - 1;
    const uint64_t bd = xor3(jd[j], si[j], new0), bu0 = ju[j] ^ si[j];
    F[j] = zmap{eval(g64[j], q[j], si[j], bd, bu0), eval(g64[j], q[j], si[j], bd, ~bu0)};
  }
  // the segment's map: F[S-1] o ... o F[0]
  zmap M = F[0];
#pragma unroll
  for (int j = 1; j < S; ++j) M = zcompose(F[j], M);
  // inclusive scan over the column's G lanes (C apart): segment g ends with
  // G_g o ... o G_0, a constant map (G_0 is one), i.e. the new word of its last plane
  for (int d = 1; d < G; d *= 2) {
    const zmap T{shfl_up64(M.f0, d * C, 64), shfl_up64(M.f1, d * C, 64)};
    if (g >= d) M = zcompose(M, T);
  }
  uint64_t v = shfl_up64(M.f0, C, 64);  // the new word below the segment's first plane
  if (!live) return;
#pragma unroll
  for (int j = 0; j < S; ++j) {
    v = (g == 0 && j == 0) ? F[0].f0 : sel(v, F[j].f1, F[j].f0);
    s[(int64_t)(z0 + j) * L2 + c0] = v;
  }
}

// one launch per colour; thread = (column, segment), grid.y = system
template <bool COUNTER, bool FAST, int S>
__global__ void __launch_bounds__(256) k_sweep3d_zscan(sweep_args p, int color, int G) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int C = 64 / G, lane = i & 63;
  const int k = (i >> 6) * C + lane % C, g = lane / C;
  const bool live = k < p.L * (p.L >> 1);
  zscan_segment<COUNTER, FAST, S>(p, color, live ? k : 0, g, G, blockIdx.y, live);
}

// ---------------------------------------------------------------- 2D half-sweep
// site k (0 <= k < L*L/2) of colour `color`, systems sys0 .. sys0+MB-1
template <bool COUNTER, bool FAST, bool OPEN, int MB>
__device__ __forceinline__ void half2d_site(const sweep_args &p, int color, int k, int sys0) {
  const int L = p.L;
  const int half = L >> 1;
  const int y = k / half;
  const int x = 2 * (k - y * half) + ((y + color) & 1);
  const int xm = x == 0 ? L - 1 : x - 1, xp = x == L - 1 ? 0 : x + 1;
  const int ym = y == 0 ? L - 1 : y - 1, yp = y == L - 1 ? 0 : y + 1;
  const int c0 = x + L * y;
  const int cw = xm + L * y, ce = xp + L * y, cn = x + L * ym, cs = x + L * yp;
  const uint64_t jw = p.jx[c0], je = p.jx[ce], jn = p.jy[c0], js = p.jy[cs];
  uint64_t g;
  if (COUNTER) {
    const u32x4 r = counter_block((uint32_t)(((x & ~3) | (x & 1)) + L * y), p.seed, p.sweep);
    g = counter_half(r, (x >> 1) & 1);
  } else {
    g = p.words[(int64_t)color * (p.N >> 1) + k];
  }
  const bool border = OPEN && (x == 0 || x == L - 1);
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    uint64_t *s = p.s + (int64_t)(sys0 + m) * p.N;
    const uint64_t si = s[c0];
    uint64_t bw = xor3(jw, si, s[cw]);
    uint64_t be = xor3(je, si, s[ce]);
    if (OPEN) {  // missing open-x bond counts as satisfied (src/cpu_2dp.cpp:338-339)
      if (x == 0) bw = ~0ULL;
      if (x == L - 1) be = ~0ULL;
    }
    const uint64_t bn = xor3(jn, si, s[cn]);
    const uint64_t bs = xor3(js, si, s[cs]);
    const count3 c = count4(bw, be, bn, bs);
    const sys_table &t = p.tab[sys0 + m];
    s[c0] = (FAST && !OPEN) ? update_fast2(t, g, c, si) : update_general(t, border ? 2 : 0, g, c, si, 5);
  }
}

template <bool COUNTER, bool FAST, bool OPEN, int MB>
__global__ void __launch_bounds__(256) k_sweep2d_half(sweep_args p, int color) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= p.L * (p.L >> 1)) return;
  half2d_site<COUNTER, FAST, OPEN, MB>(p, color, k, blockIdx.y * MB);
}

// ---------------------------------------------------------------- odd L
// With odd L the wrap neighbours in x and in y have the same colour: in a half-sweep
// the site (L-1, y) reads the new (0, y), the site (x, L-1) the new (x, 0), and
// (L-1, L-1) the new (0, L-1) and (L-1, 0) -- each is visited after its partner in
// the reference's row-major order (src/cpu_3d.cpp:94-105, src/cpu_2dp.cpp:106-114),
// which sees the partner's new value and the other way round the old one.  These
// groups (a site of the (L-1) x (L-1) corner block [0, L-1)^2 with its partners in
// the last column / last row / corner) are closed: every other neighbour of a group
// site has the other colour and does not change in the half-sweep, and along z a
// site's same-colour neighbours are its own column.  A group's sites are updated
// in visit order with the new words of its own sites passed on in registers (the
// partners' +x / +y neighbours); every other neighbour is an old word.  The corner
// block holds (L-1)^2/2 sites of each colour.  Open x (2p): the x-wrap has no bond,
// so the x partner is merely handled in the same group.

// visit rank of colour-c site (x, y) in plane z (the replay word it consumes): all
// colour-0 sites come first; a row holds (L-1)/2 sites plus one when it starts at x=0
__device__ __forceinline__ int64_t odd_rank(int L, int nz, int c, int x, int y, int z) {
  const int64_t L2 = (int64_t)L * L;
  const int64_t P0 = (L2 + 1) / 2, Pc = c ? L2 / 2 : P0;  // colour-0 / colour-c sites per plane
  const int64_t rows_before = (int64_t)y * ((L - 1) / 2) + (c == 0 ? (y + 1) / 2 : y / 2);
  return (c ? nz * P0 : 0) + z * Pc + rows_before + (x - ((y + c) & 1)) / 2;
}

// groups of one colour: (L-1)^2/2 corner-block sites, one per thread
__host__ __device__ __forceinline__ int odd_groups(int L) { return (L - 1) * ((L - 1) >> 1); }

// Group k's members: 0 = (x, y) in the corner block, 1 = (L-1, y) when x = 0, 2 = (x, L-1)
// when y = 0, 3 = (L-1, L-1) when x = y = 0.  Forwarded new words: member 1's +x
// neighbour is member 0, member 2's +y neighbour is member 0, member 3's are members 2
// (+x) and 1 (+y).
struct odd_member {
  int c0, cw, ce, cn, cs;  // in-plane offsets of the site and its -x, +x, -y, +y neighbours
};
__device__ __forceinline__ odd_member odd_offsets(int L, int x, int y) {
  const int xm = x == 0 ? L - 1 : x - 1, xp = x == L - 1 ? 0 : x + 1;
  const int ym = y == 0 ? L - 1 : y - 1, yp = y == L - 1 ? 0 : y + 1;
  return odd_member{x + L * y, xm + L * y, xp + L * y, x + L * ym, x + L * yp};
}
struct odd_loads {
  uint64_t jw, je, jn, js, jd;  // couplings: -x, +x, -y, +y, +z bonds
  uint64_t w, e, n, s, d;       // old neighbour words (e / s not loaded where forwarded)
};

// 3D: one lane per member.  Lane i of a system's odd_width(L) lanes (systems start
// at a wave boundary):
//   i < 4h (h = (L-1)/2): lane pairs (2q, 2q+1) = (corner-block site, its partner)
//     colour 0: q = 0: (0,0) & (0,L-1);  q = 1: (L-1,0) & (L-1,L-1);
//               q = 2..h: (2(q-1),0) & (2(q-1),L-1);  q = h+1..2h-1: (0,y) & (L-1,y), y = 2(q-h)
//     colour 1: q < h: (1+2q,0) & (1+2q,L-1);  q = h..2h-1: (0,y) & (L-1,y), y = 1+2(q-h)
//   then the other corner-block sites (1 <= x, y <= L-2), two rows at a time;
//   lanes from the colour's site count on are idle.
// Member 0 sites walk z in step tau = z, members 1 and 2 in tau = z+1, member 3 in
// tau = z+2: a partner updates plane z one step after the site it reads the new
// word of, which then sits in that lane's `up` register and is passed by a wave
// shuffle.  The other same-colour wrap neighbours (a member 0 site reads its
// partners, members 1 and 2 read (L-1,L-1)) are updated one step or more after the
// reader has used their old word, and all other neighbours have the other colour,
// so every lane prefetches its plane loads two steps ahead like the even walk.
__host__ __device__ __forceinline__ int odd_width(int L) { return ((L * L + 1) / 2 + 63) & ~63; }

template <bool COUNTER, bool FAST>
__device__ __forceinline__ void odd3d_lane(const sweep_args &p, int color, int i, int sys) {
  const int L = p.L, h = (L - 1) >> 1;
  const int64_t L2 = (int64_t)L * L;
  const int64_t Pc = color ? L2 / 2 : (L2 + 1) / 2;  // sites of this colour per plane
  const int lane = i & 63;
  const bool live = i < Pc;
  int x = 0, y = 0, skew = 0, srcE = lane, srcS = lane;  // lanes of the forwarded +x / +y words
  if (i < 4 * h) {
    const int q = i >> 1, r = i & 1;
    int xr = -1, yr = -1;  // row-0 pair at x = xr, or x = 0 pair at row yr
    if (color == 0) {
      if (q == 1) {  // (L-1,0) reads the new (0,0); (L-1,L-1) reads (0,L-1) and (L-1,0)
        x = L - 1;
        y = r ? L - 1 : 0;
        skew = 1 + r;
        srcE = lane - 2;
        if (r) srcS = lane - 1;
      } else if (q <= h) {
        xr = q == 0 ? 0 : 2 * (q - 1);
      } else {
        yr = 2 * (q - h);
      }
    } else {
      if (q < h) xr = 1 + 2 * q;
      else yr = 1 + 2 * (q - h);
    }
    if (xr >= 0) {  // (xr, 0) and (xr, L-1), which reads the new (xr, 0) as its +y neighbour
      x = xr;
      y = r ? L - 1 : 0;
      skew = r;
      if (r) srcS = lane - 1;
    } else if (yr >= 0) {  // (0, yr) and (L-1, yr), which reads the new (0, yr) as its +x neighbour
      x = r ? L - 1 : 0;
      y = yr;
      skew = r;
      if (r) srcE = lane - 1;
    }
  } else {
    // rows 1 .. L-2 in pairs; a row whose x = 0 site has this colour holds h-1
    // sites (x = 2, 4, ..), the other h (x = 1, 3, ..); row 1 is of the second kind
    // for colour 0 and of the first for colour 1
    const int sidx = i - 4 * h, r2 = sidx / (2 * h - 1), rem = sidx - r2 * (2 * h - 1);
    const int y0 = 1 + 2 * r2;
    const int n0 = color ? h - 1 : h;  // sites in row y0
    if (rem < n0) {
      y = y0;
      x = (color ? 2 : 1) + 2 * rem;
    } else {
      y = y0 + 1;
      x = (color ? 1 : 2) + 2 * (rem - n0);
    }
  }
  const odd_member o = odd_offsets(L, x, y);
  const bool fwdE = srcE != lane, fwdS = srcS != lane;
  uint64_t *s = p.s + (int64_t)sys * p.N;
  const sys_table &t = p.tab[sys];
  const int64_t rk = live ? odd_rank(L, L, color, x, y, 0) : 0;
  uint64_t own = 0, up = 0, first = 0, jzu = 0;
  if (live) {
    own = s[o.c0];
    up = s[o.c0 + (L - 1) * L2];  // old plane L-1
    jzu = p.jz[o.c0];
  }
  auto load = [&](int z, odd_loads &q) {
    if (!live || z < 0 || z >= L) return;
    const int64_t P = z * L2, Pd = z == L - 1 ? 0 : P + L2;
    q.jw = p.jx[P + o.c0];
    q.je = p.jx[P + o.ce];
    q.jn = p.jy[P + o.c0];
    q.js = p.jy[P + o.cs];
    q.jd = p.jz[Pd + o.c0];
    q.w = s[P + o.cw];
    q.n = s[P + o.cn];
    q.e = fwdE ? 0 : s[P + o.ce];
    q.s = fwdS ? 0 : s[P + o.cs];
    q.d = z == L - 1 ? 0 : s[Pd + o.c0];
  };
  u32x4 blk{0, 0, 0, 0};
  // step tau: the forwarded words are the source lanes' `up` (their new word of the
  // plane this lane updates now); plane tau-skew uses the buffer filled at tau-2
  auto step = [&](int tau, const odd_loads &cur, odd_loads &far) {
    const uint64_t fe = __shfl(up, srcE), fs = __shfl(up, srcS);
    load(tau + 2 - skew, far);
    const int z = tau - skew;
    if (!live || z < 0 || z >= L) return;
    const uint64_t si = own;
    const uint64_t down = z == L - 1 ? first : cur.d;
    const count3 c = count6(xor3(cur.jw, si, cur.w), xor3(cur.je, si, fwdE ? fe : cur.e), xor3(cur.jn, si, cur.n),
                            xor3(cur.js, si, fwdS ? fs : cur.s), xor3(jzu, si, up), xor3(cur.jd, si, down));
    uint64_t g;
    if (COUNTER) {
      if ((z & 1) == 0) blk = counter_block((uint32_t)(o.c0 + L2 * z), p.seed, p.sweep);
      g = counter_half(blk, z & 1);
    } else {
      g = p.words[rk + z * Pc];
    }
    const uint64_t sn = FAST ? update_fast3(t, g, c, si) : update_general(t, 0, g, c, si, 7);
    s[z * L2 + o.c0] = sn;
    up = sn;
    if (z == 0) first = sn;
    own = down;
    jzu = cur.jd;
  };
  odd_loads b0{}, b1{}, b2{};
  load(0 - skew, b0);
  load(1 - skew, b1);
  const int steps = L + 2;
  for (int tau = 0; tau < steps; tau += 3) {
    step(tau, b0, b2);
    if (tau + 1 < steps) step(tau + 1, b1, b0);
    if (tau + 2 < steps) step(tau + 2, b2, b1);
  }
}

template <bool COUNTER, bool FAST>
__global__ void __launch_bounds__(256) k_sweep3d_odd(sweep_args p, int color) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < odd_width(p.L)) odd3d_lane<COUNTER, FAST>(p, color, i, blockIdx.y);  // whole waves
}

// 2D: all members' words are loaded first, then updated in visit order
template <bool COUNTER, bool FAST, bool OPEN>
__device__ __forceinline__ void odd2d_group(const sweep_args &p, int color, int k, int sys) {
  const int L = p.L, h = (L - 1) >> 1;
  const int y = k / h, x = 2 * (k - y * h) + ((y + color) & 1);
  uint64_t *s = p.s + (int64_t)sys * p.N;
  const sys_table &t = p.tab[sys];
  const bool pres[4] = {true, x == 0, y == 0, x == 0 && y == 0};
  const int mx[4] = {x, L - 1, x, L - 1}, my[4] = {y, y, L - 1, L - 1};
  odd_member o[4];
  odd_loads b[4];
  uint64_t own[4], nw[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    nw[j] = 0;
    if (!pres[j]) continue;
    o[j] = odd_offsets(L, mx[j], my[j]);
    odd_loads &q = b[j];
    q.jw = p.jx[o[j].c0];
    q.je = p.jx[o[j].ce];
    q.jn = p.jy[o[j].c0];
    q.js = p.jy[o[j].cs];
    q.w = s[o[j].cw];
    q.n = s[o[j].cn];
    q.e = (j == 1 || j == 3) ? 0 : s[o[j].ce];
    q.s = (j >= 2) ? 0 : s[o[j].cs];
    own[j] = s[o[j].c0];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (!pres[j]) continue;
    const odd_loads &q = b[j];
    const int xj = mx[j], yj = my[j];
    const uint64_t si = own[j];
    const uint64_t e = j == 1 ? nw[0] : (j == 3 ? nw[2] : q.e);
    const uint64_t sv = j == 2 ? nw[0] : (j == 3 ? nw[1] : q.s);
    uint64_t bw = xor3(q.jw, si, q.w), be = xor3(q.je, si, e);
    if (OPEN) {  // missing open-x bond counts as satisfied (src/cpu_2dp.cpp:338-339)
      if (xj == 0) bw = ~0ULL;
      if (xj == L - 1) be = ~0ULL;
    }
    const count3 c = count4(bw, be, xor3(q.jn, si, q.n), xor3(q.js, si, sv));
    uint64_t g;
    if (COUNTER) {
      const u32x4 r = counter_block((uint32_t)(((xj & ~3) | (xj & 1)) + L * yj), p.seed, p.sweep);
      g = counter_half(r, (xj >> 1) & 1);
    } else {
      g = p.words[odd_rank(L, 1, color, xj, yj, 0)];
    }
    const bool border = OPEN && (xj == 0 || xj == L - 1);
    const uint64_t sn = (FAST && !OPEN) ? update_fast2(t, g, c, si) : update_general(t, border ? 2 : 0, g, c, si, 5);
    s[o[j].c0] = sn;
    nw[j] = sn;
  }
}

template <bool COUNTER, bool FAST, bool OPEN>
__global__ void __launch_bounds__(256) k_sweep2d_odd(sweep_args p, int color) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < odd_groups(p.L)) odd2d_group<COUNTER, FAST, OPEN>(p, color, k, blockIdx.y);
}

// ---------------------------------------------------------------- measure
// Per system and lane: number of satisfied -x,-y[,-z] bonds and of set spins.
//
// Memory bounds it at large ladders: every spin word once plus the couplings.  A thread
// owns one in-plane site and walks z (3D) with the word below kept in a register, so a
// plane is read by one block only (a walk over linear site indices read every plane on
// two XCDs); all system blocks of one unit (in-plane chunk, z segment) have consecutive
// slots on one XCD, which reads the unit's couplings once into its L2.
//
// Counting: per lane bit-sliced counters (bit k of plane b = bit b of lane k's count).
// Two sites at a time go through full adders into small counters; every 8 sites those
// ripple into larger ones (about 36 instructions per word; rippling each site through all
// planes and transposing every 16 sites took about 100).  At the end the block's four
// waves add their planes through LDS, and a 64x64 bit transpose across the wave (six
// butterfly stages of lane shuffles) and a popcount turn each plane into ordinary
// per-lane counts; the transposes are shared out over the waves.  One atomic per lane and
// counter and block.
//
// Measured: 32 systems of 3D L=128 (587 MB read once) 350 -> 182 us, 3.2 TB/s; one site
// per thread instead of a pair 240, units in the slots' outer order (couplings re-read by
// every system block) 210.  Three systems, as an exchange step measures: 3D L=32 29 -> 6
// us, L=128 46 -> 27, 2D L=64 14 -> 6.

// Wave-wide 64x64 bit transpose: lane i holds row i on entry, column i on exit.
// Stage d exchanges bit d of the lane index with bit d of the bit index.
__device__ __forceinline__ uint64_t wave_transpose64(uint64_t x, int lane) {
  constexpr uint64_t M32 = 0x00000000FFFFFFFFULL, M16 = 0x0000FFFF0000FFFFULL, M8 = 0x00FF00FF00FF00FFULL,
                     M4 = 0x0F0F0F0F0F0F0F0FULL, M2 = 0x3333333333333333ULL, M1 = 0x5555555555555555ULL;
#define SA_TSTAGE(D, M)                                                            \
  {                                                                                \
    const uint64_t o = __shfl_xor(x, D);                                           \
    x = (lane & D) ? ((x & ~M) | ((o & ~M) >> D)) : ((x & M) | ((o & M) << D));    \
  }
  SA_TSTAGE(32, M32)
  SA_TSTAGE(16, M16)
  SA_TSTAGE(8, M8)
  SA_TSTAGE(4, M4)
  SA_TSTAGE(2, M2)
  SA_TSTAGE(1, M1)
#undef SA_TSTAGE
  return x;
}

// The measurement's per-lane counters are kept in up to kMeasureCopies copies
// (cnt[copy][listed system][128], copy = unit index mod copies), summed on the host:
// blocks then contend for an address that much less.  A larger ladder has that many
// more addresses, and fewer copies to move and sum (32 systems: 8 copies are 131 KB).
constexpr int kMeasureCopies = 8;
__host__ __device__ __forceinline__ int measure_copies(int n) { return n <= 8 ? kMeasureCopies : 2; }

// up to four listed systems, passed by value
struct sys4 {
  int v[4];
};

// steps (sites) of one thread: 3 bonds each must stay below 2^7, one spin each below 2^6
constexpr int kMeasWalk = 40;
constexpr int kMeasE = 7, kMeasM = 6;  // planes of a thread's counters
constexpr int kMeasPlanes = kMeasE + kMeasM;

struct meas_small {  // up to 8 sites
  uint64_t e[5], m[4];
};
struct meas_big {
  uint64_t e[kMeasE], m[kMeasM];
};

// sum of two bit-sliced numbers, a += b (nb planes into na)
template <int NA, int NB>
__device__ __forceinline__ void planes_add(uint64_t (&a)[NA], const uint64_t (&b)[NB]) {
  uint64_t c = a[0] & b[0];
  a[0] ^= b[0];
#pragma unroll
  for (int i = 1; i < NA; ++i) {
    if (i < NB) {
      const uint64_t t = maj3(a[i], b[i], c);
      a[i] = xor3(a[i], b[i], c);
      c = t;
    } else {
      const uint64_t t = a[i] & c;
      a[i] ^= c;
      c = t;
    }
  }
}

// two sites' bond words (satisfied bits: sum s of weight 1, carry c of weight 2) and spins
__device__ __forceinline__ void meas_add2(meas_small &a, uint64_t s1, uint64_t c1, uint64_t w1, uint64_t s2, uint64_t c2,
                                          uint64_t w2) {
  const uint64_t c = maj3(a.e[0], s1, s2);
  a.e[0] = xor3(a.e[0], s1, s2);
  const uint64_t t = xor3(c1, c2, c), u = maj3(c1, c2, c);
  const uint64_t v = a.e[1] & t;
  a.e[1] ^= t;
  const uint64_t x = maj3(a.e[2], u, v);
  a.e[2] = xor3(a.e[2], u, v);
  const uint64_t y = a.e[3] & x;
  a.e[3] ^= x;
  a.e[4] ^= y;
  const uint64_t p = maj3(a.m[0], w1, w2);
  a.m[0] = xor3(a.m[0], w1, w2);
  const uint64_t q = a.m[1] & p;
  a.m[1] ^= p;
  const uint64_t r = a.m[2] & q;
  a.m[2] ^= q;
  a.m[3] ^= r;
}

// The block's four waves' planes summed, turned into per-lane counts and added to cnt.
template <int SB>
struct meas_shared {
  uint64_t v[2][SB][kMeasPlanes + 2][64];  // planes of two waves / the block's planes
};
//
// report (may be empty): the block that finishes last sums the copies, writes the counts to
// host memory and then `seq`, and leaves the counters and the ticket at zero for the next
// measurement -- one launch, no copy and no event per measurement (a step of a small replay
// ladder with its measurement 146 -> 116 us, 32 systems of L=128 210 -> 201).
struct meas_report {
  unsigned *ticket = nullptr;         // blocks done
  unsigned total = 0;                 // blocks in all
  int *out = nullptr;                 // host: [listed system][2][64]
  unsigned long long *flag = nullptr;  // host
  unsigned long long seq = 0;
};
template <int SB>
__device__ __forceinline__ void meas_finish(const meas_big (&big)[SB], meas_shared<SB> &sh, int (&red)[SB][2][64],
                                            int nsys, int sys0, int ns, int unit, int *cnt, const meas_report &rep) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  // the four waves' planes added through LDS: waves 2, 3 into 0, 1, then 1 into 0
  for (int q = threadIdx.x; q < SB * 128; q += blockDim.x) (&red[0][0][0])[q] = 0;
  uint64_t e[SB][kMeasE + 2], mm[SB][kMeasM + 2];
#pragma unroll
  for (int m = 0; m < SB; ++m) {
#pragma unroll
    for (int b = 0; b < kMeasE + 2; ++b) e[m][b] = b < kMeasE ? big[m].e[b < kMeasE ? b : 0] : 0;
#pragma unroll
    for (int b = 0; b < kMeasM + 2; ++b) mm[m][b] = b < kMeasM ? big[m].m[b < kMeasM ? b : 0] : 0;
  }
#pragma unroll
  for (int round = 0; round < 2; ++round) {
    const int from = round == 0 ? 2 : 1;  // waves from .. 2*from-1 hand theirs to wave - from
    if (wv >= from && wv < 2 * from) {
#pragma unroll
      for (int m = 0; m < SB; ++m) {
#pragma unroll
        for (int b = 0; b < kMeasE + 1; ++b) sh.v[wv - from][m][b][lane] = e[m][b];
#pragma unroll
        for (int b = 0; b < kMeasM + 1; ++b) sh.v[wv - from][m][kMeasE + 1 + b][lane] = mm[m][b];
      }
    }
    __syncthreads();
    if (wv < from) {
#pragma unroll
      for (int m = 0; m < SB; ++m) {
        uint64_t oe[kMeasE + 1], om[kMeasM + 1];
#pragma unroll
        for (int b = 0; b < kMeasE + 1; ++b) oe[b] = sh.v[wv][m][b][lane];
#pragma unroll
        for (int b = 0; b < kMeasM + 1; ++b) om[b] = sh.v[wv][m][kMeasE + 1 + b][lane];
        planes_add(e[m], oe);
        planes_add(mm[m], om);
      }
    }
    __syncthreads();
  }
  // wave 0's planes to all waves; each transposes its share
  constexpr int PB = kMeasPlanes + 4;  // planes per system: kMeasE + 2 and kMeasM + 2
  uint64_t *pl = &sh.v[0][0][0][0];      // [SB][PB][64]: 2 * (kMeasPlanes + 2) >= PB planes per system
  if (wv == 0) {
#pragma unroll
    for (int m = 0; m < SB; ++m) {
#pragma unroll
      for (int b = 0; b < kMeasE + 2; ++b) pl[(m * PB + b) * 64 + lane] = e[m][b];
#pragma unroll
      for (int b = 0; b < kMeasM + 2; ++b) pl[(m * PB + kMeasE + 2 + b) * 64 + lane] = mm[m][b];
    }
  }
  __syncthreads();
  for (int q = wv; q < SB * PB; q += 4) {
    const int m = q / PB, b = q - m * PB;
    const uint64_t v = pl[q * 64 + lane];
    if (__ballot(v != 0) == 0) continue;  // an empty plane
    const bool isE = b < kMeasE + 2;
    atomicAdd(&red[m][isE ? 0 : 1][lane], __popcll(wave_transpose64(v, lane)) << (isE ? b : b - kMeasE - 2));
  }
  __syncthreads();
  int *mine = cnt + ((int64_t)(unit % measure_copies(nsys)) * nsys + sys0) * 128;
  if (!rep.ticket) {
    for (int q = threadIdx.x; q < ns * 128; q += blockDim.x) atomicAdd(&mine[q], (&red[0][0][0])[q]);
    return;
  }
  // Counters, ticket and report are only touched by atomics and system-scope stores, which
  // act at the device's and the host's coherence points, so their order is all that matters,
  // not the caches' contents: an addition whose old value has come back is done, and a block
  // takes its ticket after its additions.  (A device-scope fence per block writes back and
  // invalidates the L2: measuring 32 systems of L=128 took twice as long with it.)
  __shared__ int last;
  int seen = 0;
  for (int q = threadIdx.x; q < ns * 128; q += blockDim.x) seen |= atomicAdd(&mine[q], (&red[0][0][0])[q]);
  asm volatile("" ::"v"(seen));        // the old values are used: the additions have returned
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) last = atomicAdd(rep.ticket, 1u) == rep.total - 1;
  __syncthreads();
  if (!last) return;
  const int n = nsys * 128, copies = measure_copies(nsys);
  for (int q = threadIdx.x; q < n; q += blockDim.x) {
    int v[kMeasureCopies], sum = 0;
#pragma unroll
    for (int c = 0; c < kMeasureCopies; ++c) v[c] = c < copies ? atomicExch(&cnt[(int64_t)c * n + q], 0) : 0;
#pragma unroll
    for (int c = 0; c < kMeasureCopies; ++c) sum += v[c];
    __hip_atomic_store(&rep.out[q], sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (threadIdx.x == 0) atomicExch(rep.ticket, 0u);
  // every wave's counts have left before the barrier, and the flag is a release for the host
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(rep.flag, rep.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Block = one unit (3D: 256 in-plane sites x up to `walk` planes; 2D: 256*walk
// consecutive sites) of SB systems.
template <int KIND, int SB>
__global__ void __launch_bounds__(256) k_measure(const uint64_t *__restrict__ s_all, const uint64_t *__restrict__ jx,
                                                 const uint64_t *__restrict__ jy, const uint64_t *__restrict__ jz,
                                                 int L, int64_t N, int nsys, const int *__restrict__ sys_list,
                                                 sys4 sel, int *cnt, int units, int chunks, int walk,
                                                 meas_report rep) {
  __shared__ meas_shared<SB> sh;
  __shared__ int red[SB][2][64];
  const int nq = (nsys + SB - 1) / SB;
  // blocks go round-robin over the 8 XCDs; slot i of XCD b%8: unit 8*(i/nq) + b%8, system block i%nq
  const int slot = (int)(blockIdx.x >> 3);
  const int unit = 8 * (slot / nq) + (int)(blockIdx.x & 7);
  if (unit >= units) return;
  const int sys0 = (slot % nq) * SB;
  const int ns = (nsys - sys0) < SB ? (nsys - sys0) : SB;
  const uint32_t uL = (uint32_t)L, uL2 = uL * uL;
  const uint64_t *sp[SB];
#pragma unroll
  for (int m = 0; m < SB; ++m) {
    const int q = sys0 + (m < ns ? m : 0);
    const int sys = sys_list ? sys_list[q] : (sel.v[0] >= 0 ? sel.v[q & 3] : q);  // sel: at most 4 systems
    sp[m] = s_all + (int64_t)sys * N;
  }
  // the thread's first site (x, y), its plane, and how many steps it takes
  const uint32_t p0 = (KIND == KIND_3D ? (uint32_t)(unit % chunks) * 256u : (uint32_t)unit * (uint32_t)(256 * walk)) +
                      threadIdx.x;
  uint32_t x = p0 % uL, y = p0 / uL;
  uint32_t z = KIND == KIND_3D ? (uint32_t)(unit / chunks) * (uint32_t)walk : 0u;
  const uint32_t dx = 256u % uL, dy = 256u / uL;  // 2D: the next step's site is 256 further on
  int steps;
  if (KIND == KIND_3D) {
    steps = p0 < uL2 ? min(walk, (int)(uL - z)) : 0;
  } else {
    steps = p0 < uL2 ? min(walk, (int)((uL2 - p0 + 255u) / 256u)) : 0;
  }
  const uint32_t iw0 = p0 - x + (x == 0 ? uL - 1 : x - 1), in0 = y == 0 ? p0 + uL2 - uL : p0 - uL;
  uint64_t below[SB];
#pragma unroll
  for (int m = 0; m < SB; ++m)
    below[m] = (KIND == KIND_3D && steps > 0) ? sp[m][(int64_t)(z == 0 ? uL - 1 : z - 1) * uL2 + p0] : 0;
  meas_big big[SB];
#pragma unroll
  for (int m = 0; m < SB; ++m) {
#pragma unroll
    for (int b = 0; b < kMeasE; ++b) big[m].e[b] = 0;
#pragma unroll
    for (int b = 0; b < kMeasM; ++b) big[m].m[b] = 0;
  }
  // eight steps from j0 on, four at a time with all their loads issued before any of
  // them is counted; FULL: every lane of the wave has all eight
  constexpr int U = 4;
  auto eight = [&](int j0, auto full) {
    constexpr bool FULL = decltype(full)::value;
    meas_small a[SB];
#pragma unroll
    for (int m = 0; m < SB; ++m) {
#pragma unroll
      for (int b = 0; b < 5; ++b) a[m].e[b] = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) a[m].m[b] = 0;
    }
#pragma unroll
    for (int h = 0; h < 8; h += U) {
      uint64_t Jw[U], Jn[U], Ju[U], w[U][SB], sw[U][SB], sn[U][SB];
#pragma unroll
      for (int g = 0; g < U; ++g) {
        const int j = j0 + h + g;
        const bool in = FULL || j < steps;  // steps beyond the range hold zero words and count nothing
        uint32_t i, iw, inn;
        bool west = true;
        int64_t P = 0;
        if (KIND == KIND_3D) {
          i = p0;
          iw = iw0;
          inn = in0;
          P = (int64_t)(z + (uint32_t)j) * uL2;
        } else {
          i = p0 + 256u * (uint32_t)j;
          iw = i - x + (x == 0 ? uL - 1 : x - 1);
          inn = y == 0 ? i + uL2 - uL : i - uL;
          west = !(KIND == KIND_2P && x == 0);  // no open-x west bond
          x += dx;
          y += dy;
          if (x >= uL) {
            x -= uL;
            ++y;
          }
        }
        Jw[g] = (in && west) ? jx[P + i] : 0;
        Jn[g] = in ? jy[P + i] : 0;
        Ju[g] = (in && KIND == KIND_3D) ? jz[P + i] : 0;
#pragma unroll
        for (int m = 0; m < SB; ++m) {
          w[g][m] = in ? sp[m][P + i] : 0;
          sn[g][m] = in ? sp[m][P + inn] : 0;
          // without a west bond its word is the site's own: w ^ w = 0 counts nothing
          sw[g][m] = in ? sp[m][west ? P + iw : P + i] : 0;
        }
      }
#pragma unroll
      for (int m = 0; m < SB; ++m) {
        uint64_t sb[U], cb[U];
#pragma unroll
        for (int g = 0; g < U; ++g) {
          const uint64_t bw = xor3(Jw[g], w[g][m], sw[g][m]), bn = xor3(Jn[g], w[g][m], sn[g][m]);
          if (KIND == KIND_3D) {
            const uint64_t bu = (FULL || j0 + h + g < steps) ? xor3(Ju[g], w[g][m], below[m]) : 0;
            sb[g] = xor3(bw, bn, bu);
            cb[g] = maj3(bw, bn, bu);
            below[m] = w[g][m];
          } else {
            sb[g] = bw ^ bn;
            cb[g] = bw & bn;
          }
        }
#pragma unroll
        for (int g = 0; g < U; g += 2) meas_add2(a[m], sb[g], cb[g], w[g][m], sb[g + 1], cb[g + 1], w[g + 1][m]);
      }
    }
#pragma unroll
    for (int m = 0; m < SB; ++m) {
      planes_add(big[m].e, a[m].e);
      planes_add(big[m].m, a[m].m);
    }
  };
  for (int j0 = 0; j0 < walk; j0 += 8) {
    if (__all(j0 + 8 <= steps)) eight(j0, std::true_type{});
    else eight(j0, std::false_type{});
  }
  meas_finish<SB>(big, sh, red, nsys, sys0, ns, unit, cnt, rep);
}

// 3D with an even side and spin arrays below 2^31 bytes: a thread owns a pair of
// neighbouring in-plane sites (128-bit loads; the second site's -x neighbour is the
// first), buffer loads with the plane offset in a scalar register.  A unit is 512
// in-plane sites x up to `walk` planes (walk <= kMeasWalk / 2 pairs).
template <int SB>
__global__ void __launch_bounds__(256) k_measure3d_pair(const uint64_t *__restrict__ s_all,
                                                        const uint64_t *__restrict__ jx,
                                                        const uint64_t *__restrict__ jy,
                                                        const uint64_t *__restrict__ jz, int L, int64_t N, int nsys,
                                                        const int *__restrict__ sys_list, sys4 sel, int *cnt, int units,
                                                        int chunks, int walk, meas_report rep) {
  __shared__ meas_shared<SB> sh;
  __shared__ int red[SB][2][64];
  const int nq = (nsys + SB - 1) / SB;
  const int slot = (int)(blockIdx.x >> 3);  // as in k_measure
  const int unit = 8 * (slot / nq) + (int)(blockIdx.x & 7);
  if (unit >= units) return;
  const int sys0 = (slot % nq) * SB;
  const int ns = (nsys - sys0) < SB ? (nsys - sys0) : SB;
  const uint32_t uL = (uint32_t)L, uL2 = uL * uL, bytes = (uint32_t)N * 8u;
  buf_t sp[SB];
#pragma unroll
  for (int m = 0; m < SB; ++m) {
    const int q = sys0 + (m < ns ? m : 0);
    const int sys = sys_list ? sys_list[q] : (sel.v[0] >= 0 ? sel.v[q & 3] : q);  // sel: at most 4 systems
    sp[m] = make_buf(s_all + (int64_t)sys * N, bytes);
  }
  const buf_t bx = make_buf(jx, bytes), by = make_buf(jy, bytes), bz = make_buf(jz, bytes);
  const uint32_t p0 = (uint32_t)(unit % chunks) * 512u + threadIdx.x * 2u;
  const uint32_t x = p0 % uL, y = p0 / uL;
  const int z0 = (unit / chunks) * walk, steps = min(walk, L - z0);
  const uint32_t plane = uL2 * 8u;
  // lanes beyond the plane and steps beyond the range read zeros (offset past the end)
  const bool in = p0 < uL2;
  const uint32_t vo = in ? p0 * 8u : kOutOfRange;
  const uint32_t vw = in ? (p0 - x + (x == 0 ? uL - 1 : x - 1)) * 8u : kOutOfRange;
  const uint32_t vn = in ? (y == 0 ? p0 + uL2 - uL : p0 - uL) * 8u : kOutOfRange;
  uint64_t below[SB][2];
#pragma unroll
  for (int m = 0; m < SB; ++m) bld2(sp[m], vo, (uint32_t)(z0 == 0 ? L - 1 : z0 - 1) * plane, below[m][0], below[m][1]);
  meas_big big[SB];
#pragma unroll
  for (int m = 0; m < SB; ++m) {
#pragma unroll
    for (int b = 0; b < kMeasE; ++b) big[m].e[b] = 0;
#pragma unroll
    for (int b = 0; b < kMeasM; ++b) big[m].m[b] = 0;
  }
  constexpr int U = 2;  // planes whose loads are issued together
  for (int j0 = 0; j0 < steps; j0 += 4) {
    meas_small a[SB];
#pragma unroll
    for (int m = 0; m < SB; ++m) {
#pragma unroll
      for (int b = 0; b < 5; ++b) a[m].e[b] = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) a[m].m[b] = 0;
    }
#pragma unroll
    for (int h = 0; h < 4; h += U) {
      uint64_t Jx[U][2], Jy[U][2], Jz[U][2], w[U][SB][2], sw[U][SB], sn[U][SB][2];
#pragma unroll
      for (int g = 0; g < U; ++g) {
        const int j = j0 + h + g;
        const bool ok = j < steps;  // uniform
        const uint32_t P = (uint32_t)(z0 + (ok ? j : 0)) * plane;
        const uint32_t o = ok ? vo : kOutOfRange, ow = ok ? vw : kOutOfRange, on = ok ? vn : kOutOfRange;
        bld2(bx, o, P, Jx[g][0], Jx[g][1]);
        bld2(by, o, P, Jy[g][0], Jy[g][1]);
        bld2(bz, o, P, Jz[g][0], Jz[g][1]);
#pragma unroll
        for (int m = 0; m < SB; ++m) {
          bld2(sp[m], o, P, w[g][m][0], w[g][m][1]);
          bld2(sp[m], on, P, sn[g][m][0], sn[g][m][1]);
          sw[g][m] = bld(sp[m], ow, P);
        }
      }
#pragma unroll
      for (int g = 0; g < U; ++g) {
        const uint64_t live = j0 + h + g < steps ? ~0ULL : 0ULL;
#pragma unroll
        for (int m = 0; m < SB; ++m) {
          const uint64_t w0 = w[g][m][0], w1 = w[g][m][1];
          const uint64_t x0 = xor3(Jx[g][0], w0, sw[g][m]), x1 = xor3(Jx[g][1], w1, w0);
          const uint64_t n0 = xor3(Jy[g][0], w0, sn[g][m][0]), n1 = xor3(Jy[g][1], w1, sn[g][m][1]);
          // a step beyond the range: the word below is the last plane's
          const uint64_t u0 = xor3(Jz[g][0], w0, below[m][0] & live), u1 = xor3(Jz[g][1], w1, below[m][1] & live);
          below[m][0] = w0;
          below[m][1] = w1;
          meas_add2(a[m], xor3(x0, n0, u0), maj3(x0, n0, u0), w0, xor3(x1, n1, u1), maj3(x1, n1, u1), w1);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < SB; ++m) {
      planes_add(big[m].e, a[m].e);
      planes_add(big[m].m, a[m].m);
    }
  }
  meas_finish<SB>(big, sh, red, nsys, sys0, ns, unit, cnt, rep);
}

static __global__ void k_fill_zero(int *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------- digest
// XOR over i < n of the splitmix64 finaliser of w[i] + i * golden (sa_digest with first
// index 0), into *out (zeroed by the caller).  Memory-bound: each word is read once.
static __global__ void __launch_bounds__(256) k_digest(const uint64_t *__restrict__ w, int64_t n,
                                                       unsigned long long *out) {
  uint64_t d = 0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint64_t z = w[i] + (uint64_t)i * 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    d ^= z ^ (z >> 31);
  }
#pragma unroll
  for (int s = 32; s; s >>= 1) d ^= __shfl_xor(d, s);
  __shared__ uint64_t part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = d;
  __syncthreads();
  if (threadIdx.x == 0) atomicXor(out, (unsigned long long)(part[0] ^ part[1] ^ part[2] ^ part[3]));
}

// ---------------------------------------------------------------- masked swap
// a ^= (a^b) & m, b ^= (a^b) & m (src/device.cuh:18-23)
static __global__ void __launch_bounds__(256) k_swap(uint64_t *a, uint64_t *b, uint64_t mask, int64_t N) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += stride) {
    const uint64_t va = a[i], vb = b[i];
    const uint64_t d = (va ^ vb) & mask;
    a[i] = va ^ d;
    b[i] = vb ^ d;
  }
}

// ---------------------------------------------------------------- exchange
// One exchange attempt between systems a and b from the measurement's counters: per lane
// e = float(E + h * M) of both and the lanes with -(e_a - e_b) >= min_dE swap.  Every block
// forms the mask itself (a few KB of counters) and swaps its share of the words; block 0
// records E, M and the mask in host memory.  The host's round trip per step (copy, wait,
// 64 exponentials, launch) took 10-15 us: a step of 2D L=64, 24 temperatures 46 -> 36 us, of
// 3D L=32, 16 temperatures 104 -> 93.  The kernel itself is latency: counters, mask, words.
struct exchange_args {
  uint64_t *sa, *sb;
  int64_t N, bonds;
  const int *cnt;        // [copies][n][2][64]; listed systems a, b and, if n is 3, cold
  int n, copies, cold;   // cold: its place in the list
  float min_dE;
  double ha, hb;
  int32_t *EM;           // [3][2][64]: cold, a, b
  unsigned long long *mask;
};
static __global__ void __launch_bounds__(256) k_exchange(exchange_args t) {
  __shared__ int32_t em[3][2][64];
  __shared__ uint64_t word;
  for (int q = threadIdx.x; q < t.n * 128; q += blockDim.x) {
    int64_t sum = 0;
    for (int c = 0; c < t.copies; ++c) sum += t.cnt[(int64_t)c * t.n * 128 + q];
    (&em[0][0][0])[q] = (int32_t)(2 * sum - ((q & 64) ? t.N : t.bonds));
  }
  __syncthreads();
  if (threadIdx.x < 64) {
#pragma clang fp contract(off)  // as the host rounds: product, sum, conversion
    const int k = threadIdx.x;
    const float ea = (float)((double)em[0][0][k] + t.ha * (double)em[0][1][k]);
    const float eb = (float)((double)em[1][0][k] + t.hb * (double)em[1][1][k]);
    const uint64_t m = __ballot(-(ea - eb) >= t.min_dE);
    if (k == 0) {
      word = m;
      if (blockIdx.x == 0) *t.mask = m;
    }
  }
  if (blockIdx.x == 0)
    for (int q = threadIdx.x; q < 384; q += blockDim.x) {
      const int s = q >> 7;  // cold, a, b
      t.EM[q] = (&em[s == 0 ? t.cold : s - 1][0][0])[q & 127];
    }
  __syncthreads();
  const uint64_t m = word;
  if (!m) return;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < t.N; i += stride) {
    const uint64_t va = t.sa[i], vb = t.sb[i];
    const uint64_t d = (va ^ vb) & m;
    t.sa[i] = va ^ d;
    t.sb[i] = vb ^ d;
  }
}

}  // namespace sa
