"""FP64 products of 9-point ELL matrices on the two sides of the line between
one and two rows per lane (4,297,329 and 4,301,476 rows), with holes and
without, against the same sums in numpy, bit for bit."""
import numpy as np
import pytest

from test_gpu_row_products import ell_of, inputs, row_sums, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.mark.parametrize("holes,padding", [(0, 0), (1, 1)])
@pytest.mark.parametrize("side", [2073, 2074])
def test_product_and_defect(hip, side, holes, padding):
    bands, has, x, rhs, dinv = inputs(side, np.float64, holes, True)
    s = row_sums(bands, has, x, side, range(9))
    A = ell_of(hip, bands, has, side, padding)
    assert A.q1_side == side
    xd, rd = hip.DeviceVector.from_numpy(x), hip.DeviceVector.from_numpy(rhs)
    y = hip.DeviceVector(side * side, np.float64)
    A.spmv(xd, y)
    assert np.array_equal(y.get(), run("product", s, x, rhs, dinv), equal_nan=True)
    A.spmv(xd, y, rhs=rd)
    assert np.array_equal(y.get(), run("defect", s, x, rhs, dinv), equal_nan=True)
