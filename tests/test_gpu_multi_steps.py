"""CG on many right-hand sides of a 9-point structured matrix (fused steps)
against the same solve with the structure switched off (an explicit kernel
variant: separate product, update and direction), bit for bit."""
import numpy as np
import pytest

from honei_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from honei_amd import device
    return device


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("level,R", [(2, 3), (4, 1), (5, 64), (6, 37), (8, 64)])
@pytest.mark.parametrize("var", [True, False])
def test_fused_steps_equal_separate_ones(hip, level, R, var, dtype):
    """Columns of different scales and contents, so that they stop at
    different steps (and in either direction buffer); one starts at its
    solution; caps of 0, 1, 2 and 9 steps."""
    side = P.side_of_level(level)
    n = side * side
    bands = P.diffusion_q1_bands(level)
    E = P.q1_to_ell([b.astype(dtype) for b in bands])
    g = np.random.default_rng(level * 100 + R)
    B = g.uniform(-1, 1, (n, R)) * 10.0 ** g.integers(-4, 3, R)
    for j in range(R):                       # smoother columns converge sooner
        if j % 3 == 1:
            B[:, j] = bands[4] * (1 + j)
    X0 = np.where(np.arange(R) % 2 == 0, 0.0, g.uniform(-1, 1, (n, R)))
    M = hip.EllMatrix.from_dict(E)
    assert M.q1_side == side
    Pd = hip.DeviceVector.from_numpy((1.0 / bands[4]).astype(dtype)) if var else None
    Bd = hip.DeviceVector.from_numpy(B.astype(dtype).ravel())
    for cap, eps in ((0, 1e-8), (1, 1e-8), (2, 1e-8), (9, 1e-8), (400, 1e-6 if dtype == np.float64 else 1e-3)):
        got = []
        for variant in (0, 2):
            M.set_variant(variant)
            Xd = hip.DeviceVector.from_numpy(X0.astype(dtype).ravel())
            used, rel = hip.cg_ell_multi(M, Pd, Bd, Xd, R, cap, eps, raise_on_cap=False)
            got.append((used, rel, Xd.get()))
        assert np.array_equal(got[0][0], got[1][0]), (cap, got[0][0], got[1][0])
        assert np.array_equal(got[0][1], got[1][1]), cap
        assert np.array_equal(got[0][2], got[1][2]), cap
