"""Sweeps captured from a ladder's stream: every replay moves the spins as the same sweeps run
eagerly, also with eager sweeps between the replays, for ladders that otherwise take the
LDS-resident sweeps."""
import ctypes as C

import pytest

import simulated_annealing_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,before", [
    (sa.KIND_3D, 16, 0), (sa.KIND_3D, 28, 0), (sa.KIND_3D, 28, 1), (sa.KIND_3D, 27, 1),
    (sa.KIND_2D, 64, 0), (sa.KIND_2D, 130, 1), (sa.KIND_2P, 130, 0),
])
def test_captured_sweeps(kind, L, before):
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
        if before:
            lad.sweep(before)
        lad.sync()
        lads.append(lad)
    lad, ref = lads
    t0 = lad.sweep_index
    st = C.c_void_p(sa.lib().sa_ladder_stream(lad.h))
    graph, run = C.c_void_p(), C.c_void_p()
    ok(hip.hipStreamBeginCapture(st, C.c_int(1)))
    lad.sweep(3)
    ok(hip.hipStreamEndCapture(st, C.byref(graph)))
    ok(hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    for r in range(3):
        ok(hip.hipGraphLaunch(run, st))
        lad.sync()
        ref.sweep_index = t0
        ref.sweep(3)
        for j in range(2):
            assert (lad.spins(j) == ref.spins(j)).all(), (r, j)
        for x in lads:
            x.sweep_index = 100 + r
            x.sweep(1 + r)
        for j in range(2):
            assert (lad.spins(j) == ref.spins(j)).all(), (r, j)
    ok(hip.hipGraphExecDestroy(run))
    ok(hip.hipGraphDestroy(graph))
    for x in lads:
        x.close()
