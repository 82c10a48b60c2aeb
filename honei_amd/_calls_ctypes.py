"""The entry points of csrc/pycalls.c through ctypes, for interpreters that the
module has not been built for: the same arguments, statuses and TypeErrors."""
from __future__ import annotations

from ._lib import lib, u64, vp


def _integer(o, what):
    if o is not None and not isinstance(o, int):
        raise TypeError(f"{what}: an integer or None expected, got {type(o).__name__}")
    return o or 0


def _pointers(bands):
    if len(bands) != 9:
        raise TypeError(f"nine bands expected, got {len(bands)}")
    return [_integer(b.ptr, f"band {k}") for k, b in enumerate(bands)]


def _entry(name, sizes, count, bands=None):
    """hsolve_`name` of `count` arguments: those in `sizes` are u64; argument `bands` is a list or tuple of bands, or
    the address of an array of their nine pointers, each an argument of the function."""
    f = getattr(lib(), f"hsolve_{name}")

    def call(*args):
        if len(args) != count:
            raise TypeError(f"expected {count} arguments, got {len(args)}")
        a = [_pointers(x) if i == bands and isinstance(x, (list, tuple)) else _integer(x, f"argument {i + 1}")
             for i, x in enumerate(args)]
        out = []
        for i, x in enumerate(a):
            if i == bands:
                out += [vp(p) for p in (x if isinstance(x, list) else (vp * 9).from_address(x))]
            else:
                out.append((u64 if i in sizes else vp)(x))
        return f(*out)

    return call


def set_vector_type(cls):
    if not isinstance(cls, type):
        raise TypeError("a type expected")


for _t in ("float", "double"):
    globals()[f"product_bmdv_q1_{_t}"] = _entry(f"product_bmdv_q1_{_t}", (3, 4), 6, 0)
    globals()[f"defect_q1_{_t}"] = _entry(f"defect_q1_{_t}", (4, 5), 7, 1)
    globals()[f"jacobi_q1_{_t}"] = _entry(f"jacobi_q1_{_t}", (5,), 7)
ell_spmv = _entry("ell_spmv", (), 5)
ell_jacobi = _entry("ell_jacobi", (), 6)
