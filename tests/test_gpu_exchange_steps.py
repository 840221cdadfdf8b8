"""Exchange steps decided on the device (sa_ladder_exchange_steps) against the oracle's
parallel tempering: more steps than one run between waits (128), two temperatures (the
coldest system always one of the pair), equal temperatures (every lane exchanges), a field
(rounded products), replay, and calls of uneven length; and bad arguments are refused."""
import ctypes as C

import numpy as np
import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,T,h,every,calls,rng", [
    (1, 6, [0.7, 1.2], 0.0, 1, [300], 1), (2, 4, [0.8, 1.1, 1.5], 0.0, 2, [1, 127, 2, 3], 1),
    (1, 8, [0.9, 0.9, 1.4], 0.0, 1, [40], 1), (0, 10, [0.6, 0.9, 1.4, 2.0], 0.27, 3, [129], 1),
    (2, 5, [0.6, 0.9, 1.4], -0.13, 1, [30], 0), (2, 16, [0.9, 1.0, 1.1, 1.2, 1.3], 0.0, 2, [20], 0)])
def test_steps_match_oracle(orc, kind, L, T, h, every, calls, rng):
    T = np.array(T)
    pt = sa.PT(kind, L, T, h, 31, every, rng)
    for n in calls:
        pt.step(n)
    got = pt.result()
    want = orc.pt_run(kind, L, T, h, 31, every, sum(calls), rng_mode=rng)
    for k in ("pairs", "us", "masks", "E", "spins"):
        assert (got[k] == want[k]).all(), k
    pt.close()


def test_bad_arguments_are_refused():
    lad = sa.Ladder(1, 8, 3)
    f = sa.lib().sa_ladder_exchange_steps
    f.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int] + [C.c_void_p] * 7

    def call(cold, a, b):
        i = lambda v: np.array([v], dtype=np.int32)  # noqa: E731
        arrs = [i(a), i(b), np.zeros(1, np.float32), np.zeros(1), np.zeros(1), np.zeros(1, np.uint64), np.zeros(384, np.int32)]
        return f(lad.h, 1, 1, cold, *[x.ctypes.data for x in arrs])

    assert call(0, 1, 2) == 0
    assert call(3, 0, 1) < 0 and call(0, 1, 3) < 0 and call(0, 2, 2) < 0
    assert f(lad.h, 1, 1, 0, None, None, None, None, None, None, None) < 0
    lad.close()
