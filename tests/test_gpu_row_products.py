"""Products, defects and Jacobi sweeps of 9-point matrices, banded and ELL:
the one-row-per-lane kernels of ordinary grids and the wide kernels of the
largest, against the same sums in numpy (every product and sum rounded in the
element type, in the kernels' order), bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q1_ORDER = [4, 0, 1, 2, 3, 5, 6, 7, 8]      # the banded product's order; ELL sums ascend


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


def offsets(side):
    return [(k // 3 - 1) * side + k % 3 - 1 for k in range(9)]


def row_sums(bands, has, x, side, order):
    n = side * side
    s = None
    with np.errstate(invalid="ignore", over="ignore"):
        for k in order:
            j = np.arange(n) + offsets(side)[k]
            ok = has[k] & (j >= 0) & (j < n)
            t = bands[k] * x[np.where(ok, j, 0)]
            s = np.where(ok, t if s is None else s + t, x.dtype.type(0) if s is None else s).astype(x.dtype)
    return s


def run(op, s, x, rhs, dinv):
    with np.errstate(invalid="ignore", over="ignore"):
        return s if op == "product" else rhs - s if op == "defect" else x + (rhs - s) * dinv


def call(hip, A, op, v, y):
    x, rhs, dinv = v
    if isinstance(A, hip.Q1Matrix):
        {"product": lambda: hip.q1_product(A, x, y), "defect": lambda: hip.q1_defect(A, rhs, x, y),
         "jacobi": lambda: hip.q1_jacobi(A, rhs, dinv, x, y)}[op]()
    else:
        {"product": lambda: A.spmv(x, y), "defect": lambda: A.spmv(x, y, rhs),
         "jacobi": lambda: A.jacobi(rhs, dinv, x, y)}[op]()


def ell_of(hip, bands, has, side, padding):
    """The stored entries of each row moved up to its first slots."""
    n = side * side
    stride = n + padding
    Aj, Ax = np.zeros((9, stride), np.uint64), np.zeros((9, stride), bands[0].dtype)
    Arl = np.zeros(n, np.uint64)
    i = np.arange(n)
    for k in range(9):
        r = i[has[k]]
        Aj[Arl[r], r] = r + offsets(side)[k]
        Ax[Arl[r], r] = bands[k][r]
        Arl[r] += 1
    return hip.EllMatrix(n, n, stride, 9, 1, Aj.ravel(), Ax.ravel(), Arl)


def inputs(side, dtype, holes, special):
    g = np.random.default_rng(side * 10 + holes)
    n = side * side
    bands = [g.uniform(-1, 1, n).astype(dtype) for _ in range(9)]
    x, rhs, dinv = (g.uniform(-1, 1, n).astype(dtype) for _ in range(3))
    if special:
        x[[0, n // 2, n - 1]] = np.inf, np.nan, -np.inf
    xi, yi = np.arange(n) % side, np.arange(n) // side
    has = []
    for k in range(9):
        dy, dx = k // 3 - 1, k % 3 - 1
        ok = (xi + dx >= 0) & (xi + dx < side) & (yi + dy >= 0) & (yi + dy < side)
        has.append(ok & (g.random(n) >= 0.03) if holes and k != 4 else ok)
    return bands, has, x, rhs, dinv


@pytest.mark.parametrize("op", ["product", "defect", "jacobi"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("side", [3, 4, 5, 8, 9, 63, 64, 65, 129])
def test_banded(hip, side, dtype, op):
    """Every band entry counts, also those that wrap into the next grid row; the output may start anywhere."""
    for special in (False, True):
        bands, _, x, rhs, dinv = inputs(side, dtype, 0, special)
        s = row_sums(bands, [np.ones(side * side, bool)] * 9, x, side, Q1_ORDER)
        A = hip.Q1Matrix(bands)
        v = [hip.DeviceVector.from_numpy(q) for q in (x, rhs, dinv)]
        for off in (0, 1):
            y = hip.DeviceVector.zeros(side * side + 4, dtype)
            call(hip, A, op, v, y.view(off, side * side))
            got = y.get()
            assert np.array_equal(got[off:off + side * side], run(op, s, x, rhs, dinv), equal_nan=True), (off, special)
            assert not got[:off].any() and not got[off + side * side:].any()


@pytest.mark.parametrize("op", ["product", "defect", "jacobi"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("side", [3, 4, 5, 8, 9, 63, 64, 65, 129])
def test_ell(hip, side, dtype, op):
    """Rows with all nine slots, boundary rows and rows with holes; strides with and without padding rows; the
    automatic kernel, two rows per lane, the guarded one-row kernel, and ranges of rows."""
    n = side * side
    for holes, padding, special in ((0, 0, False), (0, 3, True), (1, 0, True), (1, 2, False)):
        bands, has, x, rhs, dinv = inputs(side, dtype, holes, special)
        want = run(op, row_sums(bands, has, x, side, range(9)), x, rhs, dinv)
        A = ell_of(hip, bands, has, side, padding)
        assert A.q1_side == side
        v = [hip.DeviceVector.from_numpy(q) for q in (x, rhs, dinv)]
        for variant in (0, 2, 4, 1):
            A.set_variant(variant)
            y = hip.DeviceVector.zeros(n + 4, dtype)
            call(hip, A, op, v, y.view(1, n))
            got = y.get()
            assert np.array_equal(got[1:n + 1], want, equal_nan=True), (holes, padding, special, variant)
            assert not got[0] and not got[n + 1:].any()
        A.set_variant(0)
        if op == "jacobi":
            continue
        for r0, r1 in ((0, 1), (1, n), (n // 2, n // 2 + 3), (2, n - 1), (n - 1, n)):
            y = hip.DeviceVector.zeros(n, dtype)
            A.spmv_rows(v[0], y, r0, r1, v[1] if op == "defect" else None)
            got = y.get()
            assert np.array_equal(got[r0:r1], want[r0:r1], equal_nan=True), (r0, r1)
            assert not got[:r0].any() and not got[r1:].any()


@pytest.mark.parametrize("form", ["banded", "ell"])
def test_first_grid_of_the_wide_kernels(hip, form):
    """8,386,816 and 8,392,609 rows, the two sides of the line between the kernels."""
    for side in (2896, 2897):
        bands, has, x, rhs, dinv = inputs(side, np.float32, 0, False)
        if form == "banded":
            s = row_sums(bands, [np.ones(side * side, bool)] * 9, x, side, Q1_ORDER)
            A = hip.Q1Matrix(bands)
        else:
            s = row_sums(bands, has, x, side, range(9))
            A = ell_of(hip, bands, has, side, 1)
        v = [hip.DeviceVector.from_numpy(q) for q in (x, rhs, dinv)]
        y = hip.DeviceVector(side * side, np.float32)
        for op in ("product", "defect", "jacobi"):
            call(hip, A, op, v, y)
            assert np.array_equal(y.get(), run(op, s, x, rhs, dinv)), (side, op)


def test_first_grid_of_the_wide_fp64_product(hip):
    """4,194,304 and 4,198,401 rows, the two sides of the FP64 product's line."""
    for side in (2048, 2049):
        bands, _, x, rhs, dinv = inputs(side, np.float64, 0, False)
        s = row_sums(bands, [np.ones(side * side, bool)] * 9, x, side, Q1_ORDER)
        A = hip.Q1Matrix(bands)
        v = [hip.DeviceVector.from_numpy(q) for q in (x, rhs, dinv)]
        y = hip.DeviceVector(side * side, np.float64)
        for op in ("product", "defect", "jacobi"):
            call(hip, A, op, v, y)
            assert np.array_equal(y.get(), run(op, s, x, rhs, dinv)), (side, op)
