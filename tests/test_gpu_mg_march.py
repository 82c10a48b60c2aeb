"""The one-pass level kernels of the multigrid engine on matrices that take
each of their storage forms and every kind of tile, against the oracle's
Multigrid<MIXED>, bit for bit: with one outer step from x0 = 0 the result is
the FP32 inner iterate itself (scale 1), which no reduction enters."""
import numpy as np
import pytest

from honei_amd import problems as P
from honei_fixtures import dinv_reference

pytestmark = pytest.mark.gpu

MINL = 2
MASKS = {6: (2,) * 8, 7: (1, 2, 1, 2, 2, 1, 1, 2), 8: (2, 2, 2, 2, 1, 2, 1, 2), 9: (1, 2, 2, 1, 2, 1, 2, 2),
         10: (2, 1, 2, 2, 2, 2, 1, 1)}


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.fixture(scope="module")
def oracle():
    from oracle.pyoracle import Oracle
    return Oracle()


def _bands(kind, level, g):
    """Nine FP32 bands, every entry non-zero (also those whose linear neighbour
    lies in the next grid row): near the interior Poisson row, by node from
      rows    7 distinct rows at random nodes (row codes, changing everywhere)
      layers  3 distinct rows by grid row, one for the most part (row codes)
      values  4 values per band at random (value codes, more than 256 rows)
      plain   continuous values (the bands themselves)."""
    side = P.side_of_level(level)
    n = side * side
    base = np.full(9, -1.0 / 3.0)
    base[4] = 8.0 / 3.0
    if kind == "plain":
        f = 1.0 + 0.05 * g.uniform(-1, 1, (9, n))
    elif kind == "values":
        f = 1.0 + 0.05 * g.uniform(-1, 1, (9, 4))[np.arange(9)[:, None], g.integers(0, 4, (9, n))]
    else:
        rows = 1.0 + 0.05 * g.uniform(-1, 1, (9, 7))
        if kind == "rows":
            at = g.integers(0, 7, n)
        else:
            at = np.repeat(np.where(np.arange(side) % 11 < 8, 0, np.arange(side) % 11 - 7), side)
        f = rows[:, at]
    return [np.ascontiguousarray((base[k] * f[k]).astype(np.float32)) for k in range(9)]


@pytest.mark.parametrize("kind", ["rows", "layers", "values", "plain"])
@pytest.mark.parametrize("level", [6, 7, 8, 9, 10])
def test_one_outer_step_equals_oracle(hip, oracle, level, kind):
    """65^2 and 129^2: one and two strips, all of them at the grid's ends;
    257^2 and 1025^2: tiles away from them, several tile heights."""
    g = np.random.default_rng(100 * level + len(kind))
    n = P.side_of_level(level) ** 2
    a32 = {L: _bands(kind, L, g) for L in range(MINL, level + 1)}
    d32 = {L: dinv_reference(a32[L][4]) for L in a32}
    A64 = [b.astype(np.float64) for b in a32[level]]
    b = g.uniform(-1, 1, n)
    ref = oracle.mg_mixed_q1(A64, b, np.zeros(n), a32, d32, min_level=MINL, max_level=level, mask=MASKS[level],
                             max_outer=1)
    assert np.isfinite(ref["x"]).all()
    mg = hip.MGSolver(hip.mg_params(MINL, level, mask=MASKS[level], max_outer=1), A64, a32, d32)
    bd, xd = hip.DeviceVector.from_numpy(b), hip.DeviceVector.zeros(n)
    for codes in (True, False):
        mg.set_value_codes(codes)
        xd.fill(0.0)
        info = mg.solve(bd, xd, raise_on_cap=False)
        assert (info["outer"], info["inner"]) == (ref["outer"], ref["inner"])
        assert np.array_equal(xd.get(), ref["x"]), (codes, np.count_nonzero(xd.get() != ref["x"]))


@pytest.mark.parametrize("level,minl", [(3, 1), (3, 2), (4, 1), (4, 2), (5, 2), (6, 1), (6, 3), (7, 2), (8, 4)])
def test_bottom_levels_equal_oracle(hip, oracle, level, minl):
    """The bottom-levels kernels with every number of levels below the finest,
    coarsest levels of one wave (3^2, 5^2) and larger ones."""
    g = np.random.default_rng(10 * level + minl)
    n = P.side_of_level(level) ** 2
    a32 = {L: _bands("plain", L, g) for L in range(minl, level + 1)}
    d32 = {L: dinv_reference(a32[L][4]) for L in a32}
    A64 = [b.astype(np.float64) for b in a32[level]]
    for mask in MASKS.values():
        b = g.uniform(-1, 1, n)
        ref = oracle.mg_mixed_q1(A64, b, np.zeros(n), a32, d32, min_level=minl, max_level=level, mask=mask, max_outer=1)
        assert np.isfinite(ref["x"]).all()
        mg = hip.MGSolver(hip.mg_params(minl, level, mask=mask, max_outer=1), A64, a32, d32)
        xd = hip.DeviceVector.zeros(n)
        info = mg.solve(hip.DeviceVector.from_numpy(b), xd, raise_on_cap=False)
        assert (info["outer"], info["inner"]) == (ref["outer"], ref["inner"])
        assert np.array_equal(xd.get(), ref["x"]), (mask, np.count_nonzero(xd.get() != ref["x"]))


@pytest.mark.parametrize("level,minl", [(7, 1), (8, 1), (8, 2)])
def test_bottom_up_to_65_equals_oracle(hip, oracle, level, minl):
    """The bottom kernel with 65^2 as its top level, on both coarsest levels of one wave."""
    g = np.random.default_rng(10 * level + minl)
    n = P.side_of_level(level) ** 2
    a32 = {L: _bands("plain", L, g) for L in range(minl, level + 1)}
    d32 = {L: dinv_reference(a32[L][4]) for L in a32}
    A64 = [b.astype(np.float64) for b in a32[level]]
    for mask in MASKS.values():
        b = g.uniform(-1, 1, n)
        ref = oracle.mg_mixed_q1(A64, b, np.zeros(n), a32, d32, min_level=minl, max_level=level, mask=mask, max_outer=1)
        assert np.isfinite(ref["x"]).all()
        mg = hip.MGSolver(hip.mg_params(minl, level, mask=mask, max_outer=1), A64, a32, d32)
        xd = hip.DeviceVector.zeros(n)
        info = mg.solve(hip.DeviceVector.from_numpy(b), xd, raise_on_cap=False)
        assert (info["outer"], info["inner"]) == (ref["outer"], ref["inner"])
        assert np.array_equal(xd.get(), ref["x"]), (mask, np.count_nonzero(xd.get() != ref["x"]))


@pytest.mark.parametrize("level", [6, 9])
def test_batch_of_three_equals_single(hip, level):
    """Two slots share a workgroup's matrix loads, the third has one alone."""
    n = P.side_of_level(level) ** 2
    g = np.random.default_rng(level)
    prm = hip.mg_params(MINL, level, mask=P.DIFFUSION_MASK, max_outer=3)
    a32 = {L: P.diffusion_ell(L, dtype=np.float32) for L in range(MINL, level + 1)}
    A64 = P.diffusion_ell(level)
    mg = hip.MGSolver.from_ell(prm, A64, a32, None, slots=3)
    bs = [hip.DeviceVector.from_numpy(g.uniform(-1, 1, n)) for _ in range(3)]
    xs = [hip.DeviceVector.zeros(n) for _ in range(3)]
    mg.solve_batch(bs, xs, raise_on_cap=False)
    one = hip.DeviceVector.zeros(n)
    for b, x in zip(bs, xs):
        one.fill(0.0)
        mg.solve(b, one, raise_on_cap=False)
        assert np.array_equal(x.get(), one.get())


@pytest.mark.parametrize("S", [2, 5, 8])
def test_outer_defect_of_several_slots_equals_single(hip, S):
    """Groups of two and four slots share a workgroup's FP64 bands; the last group of five holds one.  Columns of
    different smoothness end their inner solves, and the whole solve, in different ticks."""
    level = 7
    n = P.side_of_level(level) ** 2
    g = np.random.default_rng(S)
    prm = hip.mg_params(MINL, level, mask=P.DIFFUSION_MASK)
    a32 = {L: P.diffusion_ell(L, dtype=np.float32) for L in range(MINL, level + 1)}
    A64 = P.diffusion_ell(level)
    B = [np.ones(n) if j % 3 == 1 else g.uniform(-1, 1, n) * (np.arange(n) < n // (1 + j)) for j in range(S)]
    mg = hip.MGSolver.from_ell(prm, A64, a32, slots=S)
    bd = [hip.DeviceVector.from_numpy(b) for b in B]
    xd = [hip.DeviceVector.zeros(n) for _ in B]
    infos = mg.solve_batch(bd, xd)
    one = hip.MGSolver.from_ell(prm, A64, a32)
    for j in range(S):
        x = hip.DeviceVector.zeros(n)
        info = one.solve(bd[j], x)
        assert np.array_equal(x.get(), xd[j].get()), j
        assert (info["outer"], info["inner"]) == (infos[j]["outer"], infos[j]["inner"])


@pytest.mark.parametrize("kind", ["rows", "layers", "values"])
@pytest.mark.parametrize("level", [6, 7, 8])
def test_coded_outer_defect_equals_bands(hip, level, kind):
    """The FP64 outer defect from row codes, value codes and the bands themselves: four outer steps, so that the
    defect of an iterate enters the next inner solve."""
    g = np.random.default_rng(level)
    n = P.side_of_level(level) ** 2
    a32 = {L: _bands(kind, L, g) for L in range(MINL, level + 1)}
    d32 = {L: dinv_reference(a32[L][4]) for L in a32}
    A64 = [b.astype(np.float64) for b in a32[level]]
    mg = hip.MGSolver(hip.mg_params(MINL, level, mask=MASKS[level], max_outer=4), A64, a32, d32)
    b = hip.DeviceVector.from_numpy(g.uniform(-1, 1, n))
    got = []
    for codes in (True, False):
        mg.set_value_codes(codes)
        x = hip.DeviceVector.zeros(n)
        info = mg.solve(b, x, raise_on_cap=False)
        got.append((x.get(), info))
    # (one of the matrices makes the iteration diverge, to the same NaN)
    assert np.array_equal(list(got[0][1].values()), list(got[1][1].values()), equal_nan=True)
    assert np.array_equal(got[0][0], got[1][0], equal_nan=True)
