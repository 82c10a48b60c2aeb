"""The CPython entry points (csrc/pycalls.c): arguments they refuse, and the
statuses and messages they return, those of the ctypes calls."""
import ctypes as C

import numpy as np
import pytest

from honei_amd._lib import calls, lib, u64, vp

BANDS = (vp * 9)(*range(16, 160, 16))        # addresses that no call below reads


@pytest.mark.parametrize("name,count", [("product_bmdv_q1", 6), ("defect_q1", 7), ("jacobi_q1", 7), ("ell_spmv", 5),
                                        ("ell_jacobi", 6)])
def test_refused_arguments(name, count):
    for suffix in ("",) if name.startswith("ell") else ("_float", "_double"):
        f = getattr(calls(), name + suffix)
        for bad in (1.0, "16", b"16", np.int64(16), vp(16)):
            with pytest.raises(TypeError):
                f(*[0] * (count - 1), bad)
        for n in (0, count - 1, count + 1):
            with pytest.raises(TypeError):
                f(*[0] * n)


@pytest.mark.parametrize("dtype", ["float", "double"])
def test_status_and_message(dtype):
    """Null vectors, aliased sweep vectors, a size that is no square, and the empty call."""
    L, at = lib(), C.addressof(BANDS)

    def same(mine, theirs):
        rc = mine()
        text = L.hsolve_last_error()
        assert rc == theirs() and (rc == 0 or text == L.hsolve_last_error())
        return rc

    jac, cjac = getattr(calls(), f"jacobi_q1_{dtype}"), getattr(L, f"hsolve_jacobi_q1_{dtype}")
    for a in ((None, 32, 48, 64, 9), (16, 32, 48, 48, 9), (16, 32, 48, 64, 8), (16, 32, 48, 64, 0)):
        rc = same(lambda: jac(a[0], at, *a[1:], None),
                  lambda: cjac(vp(a[0]), BANDS, vp(a[1]), vp(a[2]), vp(a[3]), u64(a[4]), vp(None)))
        assert (rc == 0) == (a[4] == 0)
    prod, cprod = getattr(calls(), f"product_bmdv_q1_{dtype}"), getattr(L, f"hsolve_product_bmdv_q1_{dtype}")
    dfct, cdfct = getattr(calls(), f"defect_q1_{dtype}"), getattr(L, f"hsolve_defect_q1_{dtype}")
    b = [vp(p) for p in BANDS]
    for x, y, n, m in ((0, 32, 9, 3), (16, 0, 9, 3), (16, 32, 9, 4), (16, 32, 0, 0)):
        same(lambda: prod(at, x, y, n, m, None), lambda: cprod(*b, vp(x), vp(y), u64(n), u64(m), vp(None)))
        same(lambda: dfct(48, at, x, y, n, m, None), lambda: cdfct(vp(48), *b, vp(x), vp(y), u64(n), u64(m), vp(None)))
        assert dfct(0, at, 16, 32, 9, 3, None) != 0
    assert same(lambda: calls().ell_spmv(0, 16, 32, None, None), lambda: L.hsolve_ell_spmv(None, vp(16), vp(32), None, None))
    assert same(lambda: calls().ell_jacobi(None, 16, 32, 48, 64, 0),
                lambda: L.hsolve_ell_jacobi(None, vp(16), vp(32), vp(48), vp(64), None))
