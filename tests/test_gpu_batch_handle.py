"""A batch instance's ladder (sa_batch_ladder) used between two runs, against the oracle bit
for bit: new couplings take effect in the next run, whichever form sweeps the instance."""
import numpy as np
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu

# 3D half-sweeps, tiles with an even and an odd side; 2D whole, bands, odd; open x
FORMS = [(2, 6), (2, 16), (2, 13), (2, 40), (1, 32), (1, 96), (1, 33), (0, 20)]


def advance(orc, kind, L, seed, s, j, T, t0, n):
    for t in range(t0, t0 + n):
        orc.sweep(kind, L, s, *j, orc.boltz(kind, T, 0.0), orc.counter_words(kind, L, seed, t))


def new_couplings(lad, kind, s, q):
    rng = np.random.default_rng(q)
    j = [rng.integers(0, 2**64, s.size, dtype=np.uint64) for _ in range(3)]
    sa.check(sa.lib().sa_ladder_set_couplings(lad, j[0], j[1], j[2].ctypes.data if kind == 2 else None), "set_couplings")
    return j


@pytest.mark.parametrize("fetch_again", [False, True])
def test_new_couplings_take_effect(orc, fetch_again):
    b = sa.Batch()
    insts = []
    for q, (kind, L) in enumerate(FORMS):
        i = b.add(kind, L, 300 + q, 100, T=[1.1])
        jx, jy, jz, s, _ = orc.init_system(kind, L, 300 + q)
        insts.append((i, kind, L, 300 + q, s, [jx, jy, jz]))
    lads = [sa.lib().sa_batch_ladder(b.b, x[0]) for x in insts]
    b.run(5)
    for i, kind, L, seed, s, j in insts:
        advance(orc, kind, L, seed, s, j, 1.1, 0, 5)
    for q, (i, kind, L, seed, s, j) in enumerate(insts):
        lad = sa.lib().sa_batch_ladder(b.b, i) if fetch_again else lads[q]
        j[:] = new_couplings(lad, kind, s, q)
    b.run(6)
    for i, kind, L, seed, s, j in insts:
        advance(orc, kind, L, seed, s, j, 1.1, 5, 6)
        assert (b.spins(i) == s).all(), (kind, L)
    b.close()
