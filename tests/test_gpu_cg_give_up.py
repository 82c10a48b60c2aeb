"""Which way a Krylov solve runs (one launch or launches), and one-launch
solves that give up waiting, in their first launch and in a later one: the
launches that follow give the bits of the one launch."""
import ctypes as C
import time

import numpy as np
import pytest

from honei_amd import problems as P
from honei_amd._lib import lib, u64
from test_gpu_cg_one_launch import _banded, _solve

pytestmark = pytest.mark.gpu

NEVER = (1 << 64) - 1
LAUNCHES, ONE, GAVE_UP = 0, 1, 2


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.fixture(autouse=True)
def _default():
    yield
    give_up_in(NEVER)


def give_up_in(launch):
    assert lib().hsolve_krylov_give_up(u64(launch)) == 0


def path():
    p = C.c_int(-1)
    assert lib().hsolve_krylov_path(C.byref(p)) == 0
    return p.value


def same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("kind", ["none", "var", "jac", "plain"])
def test_path_taken(hip, kind):
    """One launch for one lane per row and up to 524,288 rows of nine entries, 262,144 of ten to sixteen."""
    wide = (1, 2, 3, 64, 65, 66, 900)                     # 15 entries
    for n, offsets, want in ((1, (1,), ONE), (513, (1, 17), ONE), (70001, (1, 17), ONE), (524288, (1, 17), ONE),
                             (524289, (1, 17), LAUNCHES), (262144, wide, ONE), (262145, wide, LAUNCHES),
                             (70001, wide + (950,), LAUNCHES)):
        (one, two), dinv = _banded(n, offsets, np.float64, 1)
        b = np.ones(n)
        _solve(hip, kind, hip.EllMatrix.from_dict(one), dinv, b, 3, 1e-12)
        assert path() == want, (n, offsets)
        _solve(hip, kind, hip.EllMatrix.from_dict(two), dinv, b, 3, 1e-12)
        assert path() == LAUNCHES, (n, offsets)


@pytest.mark.parametrize("kind", ["none", "var", "jac", "plain"])
def test_first_launch_gives_up(hip, kind):
    n = 70001
    (one, two), dinv = _banded(n, (1, 17, 300), np.float64, 2)
    b = np.random.default_rng(2).uniform(-1, 1, n)
    M = hip.EllMatrix.from_dict(one)
    ref = _solve(hip, kind, hip.EllMatrix.from_dict(two), dinv, b, 25, 1e-12)
    give_up_in(0)
    assert same(_solve(hip, kind, M, dinv, b, 25, 1e-12), ref) and path() == GAVE_UP
    give_up_in(NEVER)
    assert same(_solve(hip, kind, M, dinv, b, 25, 1e-12), ref) and path() == ONE


@pytest.mark.parametrize("kind", ["none", "jac"])
def test_later_launch_gives_up(hip, kind):
    """40,000 iterations (with eps 0 a solve runs to its cap), three launches of at most 16,384: the second and the
    third find the workspace of the one before advanced."""
    n = 700
    (one, two), dinv = _banded(n, (1, 26), np.float64, 3)
    b = np.random.default_rng(3).uniform(-1, 1, n)
    M = hip.EllMatrix.from_dict(one)
    ref = _solve(hip, kind, hip.EllMatrix.from_dict(two), dinv, b, 40000, 0.0)
    for launch, want in ((1, GAVE_UP), (2, GAVE_UP), (3, ONE)):
        give_up_in(launch)
        got = _solve(hip, kind, M, dinv, b, 40000, 0.0)
        assert path() == want
        assert got[0][0] == ref[0][0] == 40000 and np.array_equal(got[1], ref[1], equal_nan=True), launch


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("side", [23, 129, 363, 600, 724])
def test_banded_one_launch_equals_launches(hip, side, dtype):
    """One to four rows per thread on Q1 bands."""
    n = side * side
    A = hip.Q1Matrix([x.astype(dtype) for x in P.poisson_q1_bands(n)])
    b = hip.DeviceVector.from_numpy(P.rhs_uniform(n).astype(dtype))

    def solve():
        x = hip.DeviceVector.zeros(n, dtype)
        return hip.cg_q1(A, b, x, 30, 1e-30, raise_on_cap=False), x.get()

    one = solve()
    assert path() == ONE
    give_up_in(0)
    assert same(solve(), one) and path() == GAVE_UP


@pytest.mark.parametrize("n", [513, 70001, 524288])
def test_giving_up_takes_milliseconds_and_pauses(hip, n):
    """A wait ends after about 10 ms, and the device's next 32 solves do not try."""
    (one, two), dinv = _banded(n, (1, 17), np.float64, 4)
    b = np.random.default_rng(4).uniform(-1, 1, n)
    M = hip.EllMatrix.from_dict(one)
    ref = _solve(hip, "none", hip.EllMatrix.from_dict(two), dinv, b, 25, 1e-12)
    give_up_in(0)
    t = time.perf_counter()
    assert same(_solve(hip, "none", M, dinv, b, 25, 1e-12), ref) and path() == GAVE_UP
    assert time.perf_counter() - t < 0.1
    for _ in range(32):
        assert same(_solve(hip, "none", M, dinv, b, 25, 1e-12), ref) and path() == LAUNCHES
    _solve(hip, "none", M, dinv, b, 25, 1e-12)
    assert path() == GAVE_UP
    give_up_in(NEVER)
    _solve(hip, "none", M, dinv, b, 25, 1e-12)
    assert path() == ONE
