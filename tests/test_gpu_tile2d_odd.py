"""Odd 2D sides held whole in LDS (sa_tile2d.hpp) against the oracle, bit for bit: the smallest
sides, last groups of one and of three columns, the largest side with one item per thread (63),
the largest held at all (89) and the next one, which is not; counter and replay streams,
symmetric, general and open tables, changing temperatures."""
import numpy as np
import pytest

import simulated_annealing_amd as sa
from test_gpu_tile2d import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [sa.KIND_2D, sa.KIND_2P])
@pytest.mark.parametrize("rng", [sa.RNG_COUNTER, sa.RNG_REPLAY])
@pytest.mark.parametrize("L,nsys,nsw", [(3, 2, 70), (5, 3, 7), (7, 2, 3), (9, 1, 3), (33, 3, 5), (63, 2, 3), (65, 2, 3),
                                        (87, 1, 2), (89, 2, 3), (91, 1, 2)])
def test_odd_sides(orc, kind, rng, L, nsys, nsw):
    compare(orc, kind, L, nsys, nsw, rng, [0.6, 1.3, 2.1], [0.0, 0.0, 0.0])
    compare(orc, kind, L, nsys, min(nsw, 3), rng, [0.6, 1.3, 2.1], [0.15, 0.0, 1.5], steps=[1] * min(nsw, 3))


def test_odd_anneal(orc):
    """several sweeps per launch at changing temperatures"""
    L, nsw = 37, 9
    T = np.linspace(2.0, 0.4, nsw)
    lad = sa.Ladder(sa.KIND_2D, L, 1)
    lad.set_rng(sa.RNG_COUNTER)
    lad.seed_like_main(40)
    lad.anneal(T)
    jx, jy, jz, s, _ = orc.init_system(sa.KIND_2D, L, 40)
    for t in range(nsw):
        orc.sweep(sa.KIND_2D, L, s, jx, jy, jz, orc.boltz(sa.KIND_2D, T[t], 0.0), orc.counter_words(sa.KIND_2D, L, 40, t))
    assert (lad.spins(0) == s).all()
    lad.close()
