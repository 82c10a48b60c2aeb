"""Banded products, defects and sweeps on the two sides of the line between the
one-row-per-lane and the wide kernels (3,396,649 and 3,400,336 FP64 rows,
4,498,641 and 4,502,884 FP32 rows), with aligned and unaligned outputs, against
the same sums in numpy, bit for bit."""
import numpy as np
import pytest

from test_gpu_row_products import Q1_ORDER, call, inputs, row_sums, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.mark.parametrize("side,dtype", [(1843, np.float64), (1844, np.float64), (2121, np.float32),
                                        (2122, np.float32)])
def test_both_sides(hip, side, dtype):
    n = side * side
    for special in (False, True):
        bands, _, x, rhs, dinv = inputs(side, dtype, 0, special)
        s = row_sums(bands, [np.ones(n, bool)] * 9, x, side, Q1_ORDER)
        A = hip.Q1Matrix(bands)
        v = [hip.DeviceVector.from_numpy(q) for q in (x, rhs, dinv)]
        y = hip.DeviceVector.zeros(n + 4, dtype)
        for off in (0, 1):
            for op in ("product", "defect", "jacobi"):
                y.fill(0.0)
                call(hip, A, op, v, y.view(off, n))
                got = y.get()
                assert np.array_equal(got[off:off + n], run(op, s, x, rhs, dinv), equal_nan=True), (op, off, special)
                assert not got[:off].any() and not got[off + n:].any()
