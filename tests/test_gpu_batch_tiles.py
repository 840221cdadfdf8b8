"""Batch instances swept as LDS tiles against the oracle, bit for bit.

Sides on either side of each form's range (3D: 7 half-sweeps, 8 the smallest tile, odd ones
from 9, 64 / 65 the largest 8-column tiles, 128 / 129; 2D: 64 the largest held whole, 66
bands, 254 / 256 bands of two sweeps, 258 half-sweeps), several systems, and instances
that end inside a visit of four sweeps; chunk lengths that leave whole and partial visits;
few instances (small tiles) and many (large ones); parallel-tempering instances between."""
import numpy as np
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu

SIDES = [(2, 7), (2, 8), (2, 9), (2, 11), (2, 13), (2, 16), (2, 31), (2, 36), (2, 64), (2, 65), (1, 4), (1, 62), (1, 64),
         (1, 66), (1, 96), (1, 130), (1, 254), (1, 258), (1, 33), (0, 20)]


def final_spins(orc, kind, L, seed, T, nsw, h=0.0):
    jx, jy, jz, s, _ = orc.init_system(kind, L, seed)
    for t in range(nsw):
        orc.sweep(kind, L, s, jx, jy, jz, orc.boltz(kind, T[min(t, len(T) - 1)], h), orc.counter_words(kind, L, seed, t))
    return s


@pytest.mark.parametrize("chunk,runs", [(0, [11]), (1, [11]), (3, [11]), (5, [4, 7]), (7, [11]), (32, [1, 2, 8])])
def test_batch_tiles_match_oracle(orc, chunk, runs):
    b = sa.Batch()
    if chunk:
        b.tune(sa.TUNE_BATCH_CHUNK, chunk)
    insts = []
    for q, (kind, L) in enumerate(SIDES):
        nsw = 11 - q % 3
        T = sa.linear_schedule(2.5, 0.4, nsw)
        insts.append((b.add(kind, L, 50 + q, nsw, schedule=T), kind, L, 50 + q, T, nsw))
    two = b.add(2, 12, 7, 9, T=[0.7, 1.8], nsys=2)
    pt = b.add_pt(2, 10, [0.6, 0.9, 1.4], 77, 3, 3)
    for n in runs:
        b.run(n)
    b.run()
    for i, kind, L, seed, T, nsw in insts:
        assert b.sweeps_done(i) == nsw
        assert (b.spins(i) == final_spins(orc, kind, L, seed, T, nsw)).all(), (kind, L)
    for j, T in enumerate([0.7, 1.8]):
        assert (b.spins(two, j) == final_spins(orc, 2, 12, 7, [T], 9)).all()
    want = orc.pt_run(2, 10, np.array([0.6, 0.9, 1.4]), 0.0, 77, 3, 3, rng_mode=1)
    for j in range(3):
        assert (b.spins(pt, j) == want["spins"][j]).all()
    assert (b.pt_result(pt)["masks"] == want["masks"]).all()
    b.close()


def test_batch_large_tiles_and_limits(orc):
    """enough 3D columns for 8 x 8 tiles; the largest sides; an instance with a field between"""
    b = sa.Batch()
    insts = [(b.add(2, L, 900 + q, 2, T=[1.1]), L, 900 + q) for q, L in enumerate([128, 127, 129, 48, 47, 40])]
    fld = b.add(2, 14, 5, 2, T=[1.1], h=0.3)
    assert b.run() == 0
    for i, L, seed in insts:
        assert (b.spins(i) == final_spins(orc, 2, L, seed, [1.1], 2)).all(), L
    assert (b.spins(fld) == final_spins(orc, 2, 14, 5, [1.1], 2, 0.3)).all()
    lad = sa.lib().sa_batch_ladder(b.b, insts[3][0])  # the ladder goes on by itself
    sa.check(sa.lib().sa_ladder_sweep(lad, 3), "sweep")
    assert (b.spins(insts[3][0]) == final_spins(orc, 2, 48, 903, [1.1], 5)).all()
    b.close()
