"""CG on banded FP64 systems on the two sides of the line between guarded and
unguarded rows (1,572,516 and 1,575,025 rows) against the oracle, whose sums
run in another order: ten steps of rounding, 1e-16 each on sums of 1.6 million
terms (at most 1e-10 of the iterate's norm)."""
import numpy as np
import pytest

from honei_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [1254, 1255])
def test_ten_steps_match_oracle(hip, oracle, side):
    n = side * side
    bands = P.poisson_q1_bands(n)
    b = P.rhs_uniform(n)
    xr, it, _ = oracle.cg_none_q1(bands, b, np.zeros(n), 10, 1e-30)
    xd = hip.DeviceVector.zeros(n)
    used, _ = hip.cg_q1(hip.Q1Matrix(bands), hip.DeviceVector.from_numpy(b), xd, 10, 1e-30, raise_on_cap=False)
    assert used == it == 10
    assert np.linalg.norm(xd.get() - xr) <= 1e-10 * np.linalg.norm(xr)
