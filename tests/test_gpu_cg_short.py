"""Krylov solves of a few iterations: capped at one or none by launches, at more
in one launch."""
import numpy as np
import pytest

from test_gpu_cg_give_up import LAUNCHES, NEVER, ONE, give_up_in, path, same
from test_gpu_cg_one_launch import _banded, _solve

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.mark.parametrize("kind", ["none", "var", "jac", "plain"])
@pytest.mark.parametrize("n", [5, 300, 70001])
def test_few_iterations(hip, n, kind):
    (one, two), dinv = _banded(n, (1, 3), np.float64, 9)
    b = np.random.default_rng(9).uniform(-1, 1, n)
    M, T = hip.EllMatrix.from_dict(one), hip.EllMatrix.from_dict(two)
    give_up_in(NEVER)
    for cap in (0, 1, 2, 3, 5):
        ref = _solve(hip, kind, T, dinv, b, cap, 1e-30)
        assert same(_solve(hip, kind, M, dinv, b, cap, 1e-30), ref), cap
        assert path() == (ONE if cap >= 2 else LAUNCHES), cap
