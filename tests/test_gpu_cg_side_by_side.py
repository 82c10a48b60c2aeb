"""Krylov solves of two threads, each on a stream of its own."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from honei_amd import problems as P
from honei_amd._lib import lib, u64, vp
from test_gpu_cg_give_up import LAUNCHES, NEVER, ONE, give_up_in, path, same
from test_gpu_cg_one_launch import _banded

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


def _vectors(hip, b):
    return hip.DeviceVector.from_numpy(b), hip.DeviceVector.zeros(b.size)


def _solve(entry, M, v, stream):
    used, defect = u64(), C.c_double()
    getattr(lib(), entry)(vp(M.handle), vp(v[0].ptr), vp(v[1].ptr), u64(100), 1e-12, C.byref(used), C.byref(defect),
                          stream)
    return used.value, defect.value


@pytest.mark.parametrize("n,want", [(30000, ONE), (66049, ONE), (262144, LAUNCHES)])
def test_a_solve_does_not_wait_for_another_thread(hip, n, want):
    """The first thread's solve stands behind most of a second of other work on its stream; the second thread's, on a
    stream of its own, ends meanwhile.  Two of 30,000 rows run side by side in one launch each, of 66,049 rows the
    second with two rows a thread; 262,144 rows take every CU, so the second goes by launches."""
    (one, _), dinv = _banded(n, (1, 150), np.float64, 8)
    b = np.random.default_rng(8).uniform(-1, 1, n)
    M = hip.EllMatrix.from_dict(one)
    give_up_in(NEVER)
    v = [_vectors(hip, b) for _ in range(3)]
    ref = (_solve("hsolve_cg_ell", M, v[2], None), v[2][1].get())
    side = 129
    A = hip.Q1Matrix(P.poisson_q1_bands(side * side))
    rhs, y = hip.DeviceVector.from_numpy(P.rhs_uniform(side * side)), hip.DeviceVector.zeros(side * side)
    it = hip.DeviceVector(1, np.uint64)
    streams = [vp(), vp()]
    for st in streams:
        assert lib().hsolve_stream_create(C.byref(st)) == 0
    got, ended = {}, {}

    def first():
        for _ in range(2):      # (one workgroup, 0.4 s each)
            assert lib().hsolve_cg_konv_q1_double(A.ptrs, vp(rhs.ptr), vp(y.ptr), u64(side * side), 0.0, u64(100),
                                                  vp(it.ptr), streams[0]) == 0
        got[0], ended[0] = (_solve("hsolve_cg_ell", M, v[0], streams[0]), path()), time.perf_counter()

    def second():               # (an entry that frees no memory, which would wait for the whole device)
        got[1], ended[1] = (_solve("hsolve_cg_ell_noalloc", M, v[1], streams[1]), path()), time.perf_counter()

    began = time.perf_counter()
    a = threading.Thread(target=first)
    a.start()
    time.sleep(0.1)
    z = threading.Thread(target=second)
    z.start()
    for t in (a, z):
        t.join()
    for t, way in ((0, ONE), (1, want)):
        assert same((got[t][0], v[t][1].get()), ref) and got[t][1] == way, t
    assert ended[0] - began > 0.2, "the work ahead of the first solve was too short to tell"
    assert ended[1] < ended[0] - 0.02, (ended[1] - began, ended[0] - began)
    for st in streams:
        assert lib().hsolve_stream_destroy(st) == 0
