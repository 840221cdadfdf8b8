"""The 3D tile sweep at the limits of what the automatic choice gives it, against the oracle bit
for bit: a ladder of more systems than one launch takes (87 GB of spin arrays), and the largest sides
(up to 256; above 213 only tiles of 4 x 4 columns fit LDS, with up to 64 segments per column)."""
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu


def swept(orc, L, seed, fields):
    """a sweep at T = 1 in each field, one after the other"""
    jx, jy, jz, s, _ = orc.init_system(sa.KIND_3D, L, seed)
    for t, h in enumerate(fields):
        orc.sweep(sa.KIND_3D, L, s, jx, jy, jz, orc.boltz(sa.KIND_3D, 1.0, h), orc.counter_words(sa.KIND_3D, L, seed, t))
    return s


def test_more_systems_than_one_launch(orc):
    L, nsys = 247, 361  # 62 x 62 tiles: 360 systems a launch
    lad = sa.Ladder(sa.KIND_3D, L, nsys)
    lad.set_rng(sa.RNG_COUNTER)
    lad.seed_like_main(9)  # every system at T = 1 from the same spins
    assert lad.tuning(sa.TUNE_SWEEP3D_KERNEL) == 4
    lad.sweep(1)
    want = swept(orc, L, 9, [0.0])
    for j in (0, 1, 359, 360):
        assert (lad.spins(j) == want).all(), j
    lad.close()


@pytest.mark.parametrize("L", [200, 213, 215, 254, 255, 256])
def test_largest_sides(orc, L):
    print("[case] 3D L", L, flush=True)
    lad = sa.Ladder(sa.KIND_3D, L, 1)
    lad.set_rng(sa.RNG_COUNTER)
    lad.seed_like_main(L)
    for h in (0.0, 0.2):  # symmetric tables, then general ones
        lad.set_temperature(0, 1.0, h)
        assert lad.tuning(sa.TUNE_SWEEP3D_KERNEL) == 4
        lad.sweep(1)
    assert (lad.spins(0) == swept(orc, L, L, [0.0, 0.2])).all()
    lad.close()
