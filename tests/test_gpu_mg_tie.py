"""The multigrid engine's inner stopping test next to a tie: the tolerance at
which a solve turns from two cycles into one is the same float, and the
solution the same bits, alone, in batches and from codes and plain bands,
whose sums of the defect group the nodes differently."""
import numpy as np
import pytest

from honei_amd import problems as P

pytestmark = pytest.mark.gpu

MINL = 2


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.mark.parametrize("initial_zero", [True, False])
@pytest.mark.parametrize("level", [6, 7, 9])
def test_same_cycles_next_to_a_tie(hip, level, initial_zero):
    n = P.side_of_level(level) ** 2
    g = np.random.default_rng(level)
    A64 = P.q1_to_ell(P.poisson_q1_bands(n))
    a32 = {}
    for L in range(MINL, level + 1):
        a32[L] = P.q1_to_ell(P.poisson_q1_bands(P.side_of_level(L) ** 2))
        a32[L]["Ax"] = a32[L]["Ax"].astype(np.float32)
    b = [hip.DeviceVector.from_numpy(g.uniform(-1, 1, n)) for _ in range(2)]

    def solver(bits):
        tol = float(np.array(bits, np.uint32).view(np.float32))
        return hip.MGSolver.from_ell(hip.mg_params(MINL, level, tolerance=tol, max_outer=1, initial_zero=initial_zero),
                                     A64, a32, slots=8)

    def solve(mg, count):
        """`count` right-hand sides, the first the one that is looked at; its cycles and solution."""
        xs = [hip.DeviceVector.zeros(n) for _ in range(count)]
        infos = mg.solve_batch([b[min(i, 1)] for i in range(count)], xs, raise_on_cap=False)
        return infos[0]["inner"], xs[0].get()

    lo, hi = (int(np.float32(t).view(np.uint32)) for t in (1e-6, 0.9))
    assert (solve(solver(lo), 1)[0], solve(solver(hi), 1)[0]) == (2, 1)
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if solve(solver(mid), 1)[0] == 1 else (mid, hi)
    # (100 units in the last place lie inside the range whose sums are formed again, 1000 outside)
    for bits in (hi - 1000, hi - 100, hi - 2, hi - 1, hi, hi + 1, hi + 100, hi + 1000):
        mg = solver(bits)
        ref = solve(mg, 1)
        assert ref[0] == (1 if bits >= hi else 2)
        for codes in (True, False):
            mg.set_value_codes(codes)
            for count in (1, 2, 3, 8):
                got = solve(mg, count)
                assert got[0] == ref[0] and np.array_equal(got[1], ref[1]), (bits - hi, codes, count)
