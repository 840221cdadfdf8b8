"""An allocation that the device refuses (a ladder larger than its memory) is an error of that
call alone: ladders and batches made before go on as if it had not been made."""
import numpy as np
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu

TOO_LARGE = (sa.KIND_3D, 1024, 200)  # 1.7 TB of spins


def refused(make):
    with pytest.raises(sa.SAError) as e:
        make()
    return str(e.value)


def test_ladder_goes_on_after_a_refused_one(orc):
    L, seed = 64, 3
    lad = sa.Ladder(sa.KIND_2D, L, 2)
    lad.set_rng(sa.RNG_COUNTER)
    lad.seed_like_main(seed)
    assert "memory" in refused(lambda: sa.Ladder(*TOO_LARGE))
    lad.sweep(3)
    assert "memory" in refused(lambda: sa.Ladder(*TOO_LARGE))
    E, M = lad.measure()
    assert "memory" in refused(lambda: sa.Ladder(*TOO_LARGE))
    lad.swap(0, 1, 0xFF)
    jx, jy, jz, s, _ = orc.init_system(sa.KIND_2D, L, seed)
    for t in range(3):
        orc.sweep(sa.KIND_2D, L, s, jx, jy, jz, orc.boltz(sa.KIND_2D, 1.0, 0.0), orc.counter_words(sa.KIND_2D, L, seed, t))
    assert (lad.spins(1) == s).all()
    lad.close()


def test_batch_goes_on_after_a_refused_instance(orc):
    """... and keep their tiles' arrays, which would not have made room for it"""
    b = sa.Batch()
    T = np.array([0.6, 0.9, 1.4])
    insts = [(b.add_pt(2, 12, T, 70, 2, 9), 2, 12, 70), (b.add_pt(1, 96, T, 71, 2, 9), 1, 96, 71)]
    b.run(5)
    held = b.bytes()
    refuse = lambda: refused(lambda: b.add(*TOO_LARGE[:2], 1, 10, T=[1.0] * TOO_LARGE[2], nsys=TOO_LARGE[2]))  # noqa: E731
    assert "memory" in refuse()
    b.run(6)
    assert "memory" in refuse()
    assert b.bytes() == held
    assert b.run() == 0
    for i, kind, L, seed in insts:
        want = orc.pt_run(kind, L, T, 0.0, seed, 2, 9, rng_mode=1)
        assert (b.pt_result(i)["masks"] == want["masks"]).all(), (kind, L)
        for j in range(3):
            assert (b.spins(i, j) == want["spins"][j]).all(), (kind, L, j)
    b.close()
