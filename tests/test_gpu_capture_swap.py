"""A swap captured from a ladder's stream: every replay exchanges the lanes of the current spins,
also after eager sweeps that otherwise leave them in the other array."""
import ctypes as C

import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu

MASK = 0x00FF00FF0F0F3333


@pytest.mark.parametrize("kind,L,before", [(sa.KIND_3D, 28, 0), (sa.KIND_3D, 28, 1), (sa.KIND_3D, 27, 0),
                                           (sa.KIND_2D, 130, 0), (sa.KIND_2P, 130, 1), (sa.KIND_2D, 64, 0)])
def test_captured_swap(kind, L, before):
    hip = sa.lib()  # the HIP runtime the library is linked to, found through its handle

    def ok(e):
        assert e == 0, e

    lads = []
    for _ in range(2):
        lad = sa.Ladder(kind, L, 2)
        lad.set_rng(sa.RNG_COUNTER)
        lad.seed_like_main(5 + L)
        lad.set_temperature(0, 0.7)
        lad.set_temperature(1, 1.4)
        lad.set_spins(1, ~lad.spins(1))
        if before:
            lad.sweep(before)
        lad.sync()
        lads.append(lad)
    lad, ref = lads
    st = C.c_void_p(sa.lib().sa_ladder_stream(lad.h))
    graph, run = C.c_void_p(), C.c_void_p()
    ok(hip.hipStreamBeginCapture(st, C.c_int(1)))
    lad.swap(0, 1, MASK)
    ok(hip.hipStreamEndCapture(st, C.byref(graph)))
    ok(hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    for r in range(4):
        for x in lads:
            x.sweep(1 + r % 2)
        ok(hip.hipGraphLaunch(run, st))
        lad.sync()
        ref.swap(0, 1, MASK)
        for j in range(2):
            assert (lad.spins(j) == ref.spins(j)).all(), (r, j)
    ok(hip.hipGraphExecDestroy(run))
    ok(hip.hipGraphDestroy(graph))
    for x in lads:
        x.close()
