"""Batch instances at the largest sides of the tile forms and the first beyond, against the oracle
bit for bit: 2D bands of four sweeps up to L=256, 3D tiles up to L=128, in visits of four sweeps and
shorter ones."""
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu

SIDES = [(1, 252), (1, 254), (1, 256), (1, 258), (2, 126), (2, 127), (2, 128), (2, 129)]


@pytest.mark.parametrize("runs", [[4], [3, 2], [1, 5]])
def test_largest_sides(orc, runs):
    b = sa.Batch()
    insts = [(b.add(kind, L, 60 + q, 100, T=[0.9]), kind, L, 60 + q) for q, (kind, L) in enumerate(SIDES)]
    for n in runs:
        b.run(n)
    for i, kind, L, seed in insts:
        jx, jy, jz, s, _ = orc.init_system(kind, L, seed)
        for t in range(sum(runs)):
            orc.sweep(kind, L, s, jx, jy, jz, orc.boltz(kind, 0.9, 0.0), orc.counter_words(kind, L, seed, t))
        assert (b.spins(i) == s).all(), (kind, L)
    b.close()
