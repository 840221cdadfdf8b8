"""k_measure against plain counts: sizes at the edges of its walks and chunks.

A thread counts up to 40 sites in groups of 8 (3D: planes of a column; 2D: sites 256
apart); in-plane chunks hold 256 sites, blocks one or two systems.  The listed sizes put
the lattice below one chunk, just over one, at odd sides, at more planes than one walk and
at a partial last walk; system counts cover one and two systems per block and a last block
with one system missing."""
import numpy as np
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu


def lanes(words):
    """per-lane number of set bits of an array of words"""
    w = np.ascontiguousarray(words, dtype="<u8").reshape(-1, 1).view(np.uint8)
    return np.unpackbits(w, axis=1, bitorder="little").astype(np.int64).sum(axis=0)


def counts(kind, L, s, jx, jy, jz):
    """(E, M) per lane: 2*satisfied - bonds, 2*set - sites"""
    shape = (L, L, L) if kind == sa.KIND_3D else (1, L, L)
    v, x, y = (a.reshape(shape) for a in (s, jx, jy))
    bw = x ^ v ^ np.roll(v, 1, axis=2)
    sat = lanes(bw[:, :, 1:] if kind == sa.KIND_2P else bw) + lanes(y ^ v ^ np.roll(v, 1, axis=1))
    bonds = 2 * s.size - (L if kind == sa.KIND_2P else 0)
    if kind == sa.KIND_3D:
        sat = sat + lanes(jz.reshape(shape) ^ v ^ np.roll(v, 1, axis=0))
        bonds += s.size
    return 2 * sat - bonds, 2 * lanes(s) - s.size


@pytest.mark.parametrize("kind,L,nsys", [
    (sa.KIND_3D, 3, 1), (sa.KIND_3D, 16, 5), (sa.KIND_3D, 17, 4), (sa.KIND_3D, 41, 6), (sa.KIND_3D, 88, 9),
    (sa.KIND_2D, 3, 2), (sa.KIND_2D, 16, 1), (sa.KIND_2D, 17, 7), (sa.KIND_2D, 300, 5), (sa.KIND_2P, 129, 6),
    (sa.KIND_2P, 5, 1), (sa.KIND_2P, 1024, 3)])
def test_measure_against_counts(kind, L, nsys):
    rng = np.random.default_rng(L * 100 + nsys)
    lad = sa.Ladder(kind, L, nsys)
    n = lad.N
    draw = lambda: rng.integers(0, 1 << 64, size=n, dtype=np.uint64)  # noqa: E731
    jx, jy, jz = draw(), draw(), draw()
    lad.set_couplings(jx, jy, jz if kind == sa.KIND_3D else None)
    spins = [draw() for _ in range(nsys - 1)] + [np.full(n, ~np.uint64(0))]  # the last: every count at its largest
    for j, s in enumerate(spins):
        lad.set_spins(j, s)
    want = [counts(kind, L, s, jx, jy, jz) for s in spins]
    E, M = lad.measure()
    for j in range(nsys):
        assert (E[j] == want[j][0]).all() and (M[j] == want[j][1]).all(), j
    order = list(range(nsys))[::-1]
    E, M = lad.measure_systems(order)
    for q, j in enumerate(order):
        assert (E[q] == want[j][0]).all() and (M[q] == want[j][1]).all(), j
