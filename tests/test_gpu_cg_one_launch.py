"""Krylov solves in one launch against the same solves by
launches, bit for bit.  An ELL matrix with two lanes per row takes the
launches; with the same entries in the same order its row sums, and so its
solves, are those of the one-lane form."""
import ctypes as C
import threading

import numpy as np
import pytest

from honei_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.fixture(scope="module")
def oracle():
    from oracle.pyoracle import Oracle
    return Oracle()


def _banded(n, offsets, dtype, seed, far=None):
    """Symmetric diagonally dominant matrix with entries at +-offsets (and
    +-far, beyond 16-bit column offsets), rows ascending; two ELL layouts."""
    g = np.random.default_rng(seed)
    offs = sorted(o for o in list(offsets) + ([far] if far else []) if o < n)
    r = np.arange(n)
    cols, vals, diag = [], [], np.full(n, 0.1)
    for o in offs:
        w = -g.uniform(0.1, 1.0, n - o)
        for d, v in ((-o, np.concatenate([np.zeros(o), w])), (o, np.concatenate([w, np.zeros(o)]))):
            cols.append(np.where((r + d >= 0) & (r + d < n), r + d, n))
            vals.append(v)
            diag += np.abs(v)
    cols.append(r)
    vals.append(diag)
    c, v = np.stack(cols), np.stack(vals)
    order = np.argsort(c, axis=0, kind="stable")
    c, v = np.take_along_axis(c, order, 0), np.take_along_axis(v, order, 0)
    length = (c < n).sum(0)
    k = c.shape[0] + (c.shape[0] & 1)
    out = []
    for t in (1, 2):
        stride = 32 * ((n * t + 31) // 32)
        aj, ax = np.zeros((k // t, stride), np.uint64), np.zeros((k // t, stride), dtype)
        for s in range(c.shape[0]):
            ok = c[s] < n
            aj[s // t, (r * t + s % t)[ok]] = c[s][ok]
            ax[s // t, (r * t + s % t)[ok]] = v[s][ok].astype(dtype)
        out.append(dict(rows=n, cols=n, stride=stride, ncpr=k // t, threads=t, Aj=aj.ravel(), Ax=ax.ravel(),
                        Arl=((length + t - 1) // t).astype(np.uint64)))
    return out, (1.0 / diag).astype(dtype)


def _solve(hip, kind, M, dinv, b, iters, eps, stream=None):
    bd, xd = hip.DeviceVector.from_numpy(b), hip.DeviceVector.zeros(b.size, b.dtype)
    dd = hip.DeviceVector.from_numpy(dinv)
    if kind == "none":
        r = hip.cg_ell(M, bd, xd, iters, eps, stream=stream, raise_on_cap=False)
    elif kind == "var":
        r = hip.pcg_ell(M, dd, bd, xd, iters, eps, stream=stream, raise_on_cap=False)
    elif kind == "jac":
        r = hip.pcg_jac_ell(M, dd, bd, xd, iters, eps, stream=stream, raise_on_cap=False)
    else:
        r = hip.cg_iters_ell(M, bd, xd, iters, stream=stream)
    return r, xd.get(stream)


# block counts where the rows per thread change (256 rows a block, 512 blocks
# a row), one block and its edges, and the first size past the one launch
SIZES = [1, 2, 255, 256, 257, 513, 70001, 131072, 131073, 262144, 262145, 393217, 524288, 524289]


@pytest.mark.parametrize("kind", ["none", "var", "jac", "plain"])
@pytest.mark.parametrize("n", SIZES)
def test_one_launch_equals_launches(hip, n, kind):
    g = np.random.default_rng(n)
    for dtype, offsets, far in ((np.float64, (1, 17, 300), None), (np.float32, (1, 2, 40, 41), None),
                                (np.float64, (1, 3, 5, 64, 65, 900), 40000)):
        (one, two), dinv = _banded(n, offsets, dtype, n, far)
        b = g.uniform(-1, 1, n).astype(dtype)
        ref = _solve(hip, kind, hip.EllMatrix.from_dict(two), dinv, b, 25, 1e-12)
        got = _solve(hip, kind, hip.EllMatrix.from_dict(one), dinv, b, 25, 1e-12)
        assert got[0] == ref[0], (dtype, offsets, got[0], ref[0])
        assert np.array_equal(got[1], ref[1]), (dtype, offsets)


@pytest.mark.parametrize("kind", ["none", "jac"])
def test_more_iterations_than_one_launch_runs(hip, kind):
    """With eps 0 a solve runs to its cap, past the 16384 iterations of a launch."""
    (one, two), dinv = _banded(700, (1, 26), np.float64, 5)
    b = np.random.default_rng(6).uniform(-1, 1, 700)
    ref = _solve(hip, kind, hip.EllMatrix.from_dict(two), dinv, b, 16500, 0.0)
    got = _solve(hip, kind, hip.EllMatrix.from_dict(one), dinv, b, 16500, 0.0)
    assert got[0][0] == ref[0][0] == 16500
    assert np.array_equal(got[1], ref[1], equal_nan=True)


@pytest.mark.parametrize("side", [7, 363, 600])
def test_q1_capped_solve_matches_oracle(hip, oracle, side):
    """30 steps on Q1 bands with one, two and three rows per thread: the
    oracle's sums run in another order, so 1e-10 of the iterate's norm (30
    steps of rounding, 1e-16 each, grown by the condition 1e3 of the Krylov
    basis that far)."""
    n = side * side
    bands = P.matrix_a_bands(side)
    bands = [(x + x) * 0.5 for x in bands]
    off = P.q1_offsets(n)
    for k in range(4):          # symmetric: band -o of row i + o is band o of row i
        o = int(off[8 - k])
        bands[k][o:] = bands[8 - k][:n - o]
    b = P.rhs_uniform(n)
    xr, it, _ = oracle.cg_none_q1(bands, b, np.zeros(n), 30, 1e-30)
    xd = hip.DeviceVector.zeros(n)
    used, _ = hip.cg_q1(hip.Q1Matrix(bands), hip.DeviceVector.from_numpy(b), xd, 30, 1e-30, raise_on_cap=False)
    assert used == it
    assert np.linalg.norm(xd.get() - xr) <= 1e-10 * np.linalg.norm(xr)


def test_solves_on_two_threads_and_streams(hip):
    """Two host threads, each with its own stream and systems, give the bits
    of the same solves alone."""
    from honei_amd._lib import lib, vp
    work = []
    for t in range(2):
        (one, _), dinv = _banded(30000 + 7000 * t, (1, 150), np.float64, t)
        b = np.random.default_rng(t).uniform(-1, 1, one["rows"])
        M = hip.EllMatrix.from_dict(one)
        work.append((M, dinv, b, _solve(hip, "jac", M, dinv, b, 200, 1e-10)))
    bad = []

    def go(t):
        st = vp()
        assert lib().hsolve_stream_create(C.byref(st)) == 0
        M, dinv, b, ref = work[t]
        for _ in range(5):
            got = _solve(hip, "jac", M, dinv, b, 200, 1e-10, stream=st.value)
            if got[0] != ref[0] or not np.array_equal(got[1], ref[1]):
                bad.append(t)
        assert lib().hsolve_stream_destroy(st) == 0

    ts = [threading.Thread(target=go, args=(t,)) for t in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
