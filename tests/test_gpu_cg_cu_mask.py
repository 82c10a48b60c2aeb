"""Krylov solves on streams limited to some of the compute units: by launches,
since the one launch needs them all at once."""
import ctypes as C
import time

import numpy as np
import pytest

from honei_amd._lib import lib
from test_gpu_cg_give_up import LAUNCHES, NEVER, ONE, give_up_in, path, same
from test_gpu_cg_one_launch import _banded, _solve

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.mark.parametrize("kind", ["none", "jac"])
def test_masked_streams(hip, kind):
    runtime = lib()                             # (its symbols include those of the HIP runtime it links)
    n = 131072                                  # a workgroup on each of 256 CUs
    (one, _), dinv = _banded(n, (1, 17), np.float64, 7)
    b = np.random.default_rng(7).uniform(-1, 1, n)
    M = hip.EllMatrix.from_dict(one)
    give_up_in(NEVER)
    ref = _solve(hip, kind, M, dinv, b, 50, 1e-12)
    assert path() == ONE
    for words, want in (((0xffffffff,) * 8, ONE), ((0xffffffff,) + (0,) * 7, LAUNCHES),
                        ((0xffffffff,) * 7 + (0x7fffffff,), LAUNCHES)):
        st = C.c_void_p()
        assert runtime.hipExtStreamCreateWithCUMask(C.byref(st), C.c_uint32(8), (C.c_uint32 * 8)(*words)) == 0
        t = time.perf_counter()
        got = _solve(hip, kind, M, dinv, b, 50, 1e-12, stream=st.value)
        t = time.perf_counter() - t
        assert same(got, ref) and path() == want and t < 0.1, (words, path(), t)
        assert runtime.hipStreamDestroy(st) == 0
