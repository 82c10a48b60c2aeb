"""The bands of a Q1Matrix: products and defects read them at each call."""
import ctypes as C

import numpy as np
import pytest

from honei_amd import device
from honei_amd._lib import HsolveError, calls, vp


class Band:
    def __init__(self, ptr):
        self.ptr = ptr


@pytest.mark.parametrize("name,before", [("product_bmdv_q1_float", ()), ("product_bmdv_q1_double", ()),
                                         ("defect_q1_float", (48,)), ("defect_q1_double", (48,))])
def test_list_of_bands(name, before):
    """Lists and tuples of nine objects with a pointer; the empty call, which runs nothing and refuses null bands."""
    f = getattr(calls(), name)
    ok = [Band(p) for p in range(16, 160, 16)]
    assert f(*before, ok, 16, 32, 0, 0, None) == 0 and f(*before, tuple(ok), 16, 32, 0, 0, None) == 0
    for k in range(9):
        assert f(*before, ok[:k] + [Band(None)] + ok[k + 1:], 16, 32, 0, 0, None) == 1
    for bad, error in ((ok[:8], TypeError), (ok + ok[:1], TypeError), (ok[:8] + [Band(1.0)], TypeError),
                       (ok[:8] + [Band(vp(16))], TypeError), (ok[:8] + [16], AttributeError), (iter(ok), TypeError),
                       ({}, TypeError)):
        with pytest.raises(error):
            f(*before, bad, 16, 32, 0, 0, None)
    with pytest.raises(TypeError):
        calls().set_vector_type(16)


def test_band_pointers_follow_the_bands(monkeypatch):
    class Vector(device.DeviceVector):
        def __init__(self, ptr):
            self.buf = device._Span(None, ptr)

    made = iter(range(16, 160, 16))
    monkeypatch.setattr(device.DeviceVector, "from_numpy", classmethod(lambda cls, a: Vector(next(made))))
    A = device.Q1Matrix([np.zeros(9)] * 9)
    assert [p.value for p in A.band_ptrs()] == list(range(16, 160, 16))
    A.bands[4] = Vector(4096)
    assert A.band_ptrs()[4].value == 4096
    for gone in (Band(None), Vector(None)):
        A.bands[4] = gone
        for call in (lambda: device.q1_product(A, A.bands[0], A.bands[1]),
                     lambda: device.q1_defect(A, A.bands[0], A.bands[1], A.bands[2])):
            with pytest.raises(HsolveError, match="null"):
                call()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_replaced_band(hip, dtype):
    side = 17
    n = side * side
    g = np.random.default_rng(3)
    bands = [g.uniform(-1, 1, n).astype(dtype) for _ in range(9)]
    A, B = hip.Q1Matrix(bands), hip.Q1Matrix(bands[:5] + [2 * bands[5]] + bands[6:])
    x, r = (hip.DeviceVector.from_numpy(g.uniform(-1, 1, n).astype(dtype)) for _ in range(2))
    y, z = hip.DeviceVector(n, dtype), hip.DeviceVector(n, dtype)
    hip.q1_product(A, x, y)
    first = y.get()
    A.bands[5] = hip.DeviceVector.from_numpy(2 * bands[5])
    for call in (lambda M, out: hip.q1_product(M, x, out), lambda M, out: hip.q1_defect(M, r, x, out)):
        call(A, y)
        call(B, z)
        assert np.array_equal(y.get(), z.get()) and not np.array_equal(y.get(), first)
