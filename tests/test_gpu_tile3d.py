"""The 3D tile sweep (sa_tile3d.hpp) against the oracle, bit for bit.

Sides: the smallest; held whole in LDS (up to 26); the smallest that is not; segments of
2, 3 and 4 planes with full waves, idle lanes and a short last segment; tiles that divide
the lattice and shorter last tiles; the largest side.  Counter and replay streams,
symmetric and general tables, one sweep and several."""
import numpy as np
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu


def compare(orc, L, nsys, nsw, rng, Ts, hs, steps=None):
    kind, seed = sa.KIND_3D, 31 * L + nsys
    lad = sa.Ladder(kind, L, nsys)
    lad.set_rng(rng)
    lad.seed_like_main(seed)
    for j in range(nsys):
        lad.set_temperature(j, Ts[j], hs[j])
    for n in steps or [nsw]:
        lad.sweep(n)
    jx, jy, jz, s0, g = orc.init_system(kind, L, seed)
    ref = [s0.copy() for _ in range(nsys)]
    tabs = [orc.boltz(kind, Ts[j], hs[j]) for j in range(nsys)]
    for t in range(nsw):
        w = orc.counter_words(kind, L, seed, t) if rng == sa.RNG_COUNTER else g.fill(s0.size)
        for j in range(nsys):
            orc.sweep(kind, L, ref[j], jx, jy, jz, tabs[j], w)
    for j in range(nsys):
        assert (lad.spins(j) == ref[j]).all(), (L, j)
    lad.close()


@pytest.mark.parametrize("L", [4, 6, 8, 10, 12, 14, 16, 18, 20, 22, 24, 26, 28, 34, 36, 44, 50, 62, 64, 74, 98, 122])
def test_tile3d_counter(orc, L):
    print("[case] tile3d L", L, flush=True)
    nsys = 2 if L <= 64 else 1
    compare(orc, L, nsys, 3, sa.RNG_COUNTER, [0.6, 1.3], [0.0, 0.0], steps=[1, 2])
    compare(orc, L, nsys, 2, sa.RNG_COUNTER, [0.6, 1.3], [0.2, 1.0])


# odd sides: wrap neighbours of one colour.  Held whole up to 25; tiles from 27 on, whose last
# tile has 1 .. 7 columns; last segments of one, two and three planes
@pytest.mark.parametrize("L", [3, 5, 7, 9, 11, 13, 15, 17, 19, 21, 23, 25, 27, 29, 31, 33, 35, 37, 41, 49, 63, 71, 99])
def test_tile3d_odd_counter(orc, L):
    print("[case] tile3d odd L", L, flush=True)
    nsys = 2 if L <= 64 else 1
    compare(orc, L, nsys, 3, sa.RNG_COUNTER, [0.6, 1.3], [0.0, 0.0], steps=[1, 2])
    compare(orc, L, nsys, 2, sa.RNG_COUNTER, [0.6, 1.3], [0.2, 1.0])


@pytest.mark.parametrize("L,nsys", [(9, 33), (27, 12), (45, 8)])
def test_tile3d_odd_many_systems(orc, L, nsys):
    compare(orc, L, nsys, 3, sa.RNG_COUNTER, [0.5 + 0.1 * j for j in range(nsys)], [0.0] * nsys)


@pytest.mark.parametrize("L", [3, 4, 10, 13, 16, 27, 28, 36])
def test_tile3d_replay(orc, L):
    compare(orc, L, 2, 4, sa.RNG_REPLAY, [0.7, 1.9], [0.0, 0.0])
    compare(orc, L, 1, 3, sa.RNG_REPLAY, [0.7], [-0.3])


@pytest.mark.parametrize("L,nsys", [(8, 40), (20, 12), (40, 9)])
def test_tile3d_many_systems(orc, L, nsys):
    compare(orc, L, nsys, 3, sa.RNG_COUNTER, [0.5 + 0.1 * j for j in range(nsys)], [0.0] * nsys)


@pytest.mark.parametrize("T,h", [(0.7, 7.0), (-1.0, 0.0), (1e-3, 0.0), (1e9, 0.0), (0.9, 2.0), (0.9, -4.0)])
def test_tile3d_table_forms(orc, T, h):
    """tables with a field at and beyond the bond levels, and ones that are not compact"""
    compare(orc, 12, 2, 3, sa.RNG_COUNTER, [T, 1.0], [h, 0.0])
