"""A batch instance's ladder (sa_batch_ladder) used between two runs, against the oracle bit
for bit, whichever form sweeps the instance: new couplings take effect in the next run, and a
run goes on from the spins that sweeps and swaps of the ladder left, also through a handle that
was fetched before earlier runs."""
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


@pytest.mark.parametrize("extra", [1, 2, 3])
def test_sweeps_and_swaps_through_a_kept_handle(orc, extra):
    b = sa.Batch()
    insts = []
    for q, (kind, L) in enumerate(FORMS):
        i = b.add(kind, L, 400 + q, 100, T=[1.1, 1.1], nsys=2)
        jx, jy, jz, s, _ = orc.init_system(kind, L, 400 + q)
        insts.append((i, kind, L, 400 + q, [s, s.copy()], [jx, jy, jz], sa.lib().sa_batch_ladder(b.b, i)))
    done = 0
    for n in (5, 3, 6):
        b.run(n)
        for i, kind, L, seed, s, j, lad in insts:
            for x in s:
                advance(orc, kind, L, seed, x, j, 1.1, done, n)
        done += n
        mask = 0x0F0F0F0F0F0F0F0F << (done & 3)
        for i, kind, L, seed, s, j, lad in insts:  # the ladder's sweeps continue the instance's index
            sa.check(sa.lib().sa_ladder_set_spins(lad, 1, (~s[1])), "set_spins")
            s[1] = ~s[1]
            sa.check(sa.lib().sa_ladder_sweep(lad, extra), "sweep")
            sa.check(sa.lib().sa_ladder_swap(lad, 0, 1, mask), "swap")
            for x in s:
                advance(orc, kind, L, seed, x, j, 1.1, done, extra)
            d = (s[0] ^ s[1]) & np.uint64(mask)
            s[0] ^= d
            s[1] ^= d
    b.run(2)
    for i, kind, L, seed, s, j, lad in insts:
        for k, x in enumerate(s):
            advance(orc, kind, L, seed, x, j, 1.1, done, 2)
            assert (b.spins(i, k) == x).all(), (kind, L, k)
    b.close()
