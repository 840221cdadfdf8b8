"""sa_measure_noalloc on device arrays that start 8 bytes off a 16-byte boundary (a view into a
larger array of words), whose 3D form reads pairs of words, against sa_ladder_measure."""
import ctypes as C

import numpy as np
import pytest

import simulated_annealing_amd as sa
from test_zz_no_alloc import Hip, ladder_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,nsys", [(2, 16, 6), (2, 10, 1), (1, 32, 3), (2, 9, 2)])
@pytest.mark.parametrize("off", [[1, 1, 1, 1], [1, 0, 0, 0], [0, 1, 0, 1]])
def test_arrays_off_a_pair_boundary(kind, L, nsys, off):
    sa.lib()
    hip = Hip()
    E0, M0, s, jx, jy, jz = ladder_state(sa, kind, L, nsys, 5, 2)
    pad = np.array([0xDEADBEEFDEADBEEF], dtype=np.uint64)
    ptr = [hip.upload(np.concatenate([pad, a.reshape(-1), pad]) if o else a.reshape(-1)) + 8 * o
           for a, o in zip((s, jx, jy, jz), off)]
    junk = np.full(nsys * 64, -7, dtype=np.int32)
    dE, dM = hip.upload(junk), hip.upload(junk)
    sa.check(sa.lib().sa_measure_noalloc(kind, L, nsys, *ptr, dE, dM, None), "sa_measure_noalloc")
    hip.ok(hip.rt.hipStreamSynchronize(C.c_void_p(None)), "hipStreamSynchronize")
    E, M = hip.download(dE, junk), hip.download(dM, junk)
    hip.free()
    assert (E.reshape(nsys, 64) == E0).all() and (M.reshape(nsys, 64) == M0).all()
