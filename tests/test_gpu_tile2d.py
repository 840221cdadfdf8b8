"""2D sweeps held in LDS (sa_tile2d.hpp) against the oracle, bit for bit.

Sides: the smallest, a last group of two columns (L % 4 == 2), the largest side held whole
(88: 1936 items; 90: 2070, bands), bands that divide the lattice and a shorter last band,
halos wider than the lattice is left over, and the sides on either side of the largest one
taken.  Sweep counts: one, and more than one launch holds.  Tables: symmetric, general, and
ones that are not compact (a field larger than the bonds, a negative temperature), which
take the half-sweep kernels."""
import numpy as np
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu


def compare(orc, kind, L, nsys, nsw, rng, Ts, hs, steps=None):
    seed = 17 * L + nsys
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
        assert (lad.spins(j) == ref[j]).all(), (kind, L, j)
    lad.close()


@pytest.mark.parametrize("kind", [sa.KIND_2D, sa.KIND_2P])
@pytest.mark.parametrize("rng", [sa.RNG_COUNTER, sa.RNG_REPLAY])
@pytest.mark.parametrize("L,nsys,nsw", [(4, 1, 3), (6, 3, 70), (10, 2, 5), (64, 2, 3), (88, 1, 2), (90, 2, 7),
                                        (96, 3, 5), (130, 1, 11), (258, 2, 3), (510, 1, 2), (768, 1, 3), (770, 1, 1)])
def test_tile2d_matches_oracle(orc, kind, rng, L, nsys, nsw):
    compare(orc, kind, L, nsys, nsw, rng, [0.6, 1.3, 2.1], [0.0, 0.0, 0.0])
    compare(orc, kind, L, nsys, min(nsw, 3), rng, [0.6, 1.3, 2.1], [0.15, 0.0, 1.5])


@pytest.mark.parametrize("L,nsys", [(16, 30), (256, 20), (514, 3)])
def test_tile2d_many_systems(orc, L, nsys):
    compare(orc, sa.KIND_2D, L, nsys, 4, sa.RNG_COUNTER, [0.5 + 0.05 * j for j in range(nsys)], [0.0] * nsys,
            steps=[1, 3])


@pytest.mark.parametrize("kind", [sa.KIND_2D, sa.KIND_2P])
@pytest.mark.parametrize("T,h", [(0.7, 5.0), (-1.0, 0.0), (1e-3, 0.0), (1e9, 0.0), (0.9, -0.4), (0.9, 2.0)])
def test_tile2d_table_forms(orc, kind, T, h):
    compare(orc, kind, 22, 2, 4, sa.RNG_COUNTER, [T, 1.0], [h, 0.0])


@pytest.mark.parametrize("kind,L,nsys", [(sa.KIND_2D, 20, 2), (sa.KIND_2P, 18, 1), (sa.KIND_2D, 96, 2)])
@pytest.mark.parametrize("h", [0.0, 0.3])
@pytest.mark.parametrize("odd_one", [None, -2.0])
def test_anneal_runs_match_oracle(orc, kind, L, nsys, h, odd_one):
    """several sweeps per launch at changing temperatures; a table that is not compact
    (negative temperature) in the schedule sends the call to one sweep per launch"""
    nsw, seed = 9, 5 * L
    Ts = np.linspace(2.5, 0.3, nsw * nsys).reshape(nsw, nsys)
    if odd_one is not None:
        Ts[5, 0] = odd_one
    lad = sa.Ladder(kind, L, nsys)
    lad.set_rng(sa.RNG_COUNTER)
    lad.seed_like_main(seed)
    lad.anneal(Ts, h)
    lad.sweep(2)  # at the last temperatures
    jx, jy, jz, s0, _ = orc.init_system(kind, L, seed)
    for j in range(nsys):
        s = s0.copy()
        for t in range(nsw + 2):
            orc.sweep(kind, L, s, jx, jy, jz, orc.boltz(kind, Ts[min(t, nsw - 1), j], h), orc.counter_words(kind, L, seed, t))
        assert (lad.spins(j) == s).all(), j
    assert lad.sweep_index == nsw + 2
    lad.close()
