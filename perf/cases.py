"""Timed workloads of the sparse Poisson solver path, through the entry points
of honei_amd.device: single products, defects and smoother sweeps, Krylov
solves, multigrid solves (one and many at a time) and the request server.

Vectors are torch tensors on the GPU, handed over without a copy.  A case is a
dict of plain values; its "kind" picks one of the builders below."""
from __future__ import annotations

import math

import numpy as np
import torch

from honei_amd import device as hip

MIN_LEVEL = 2                       # coarsest level of every hierarchy (5 x 5 nodes)
TILES = 64                          # coefficient tiles per direction of the diffusion problem
LEFT_RIGHT = (2, 2, 2, 2, 1, 2, 1, 2)   # Dirichlet left and right, Neumann bottom and top

NUMPY = {"float64": np.float64, "float32": np.float32}
TORCH = {"float64": torch.float64, "float32": torch.float32}


def listed():
    return [
        # the product of the reference's headline matrix form: a 9-point stencil with coefficients of its own
        # in every row, stored as ELL, at the largest grid
        dict(name="ell_product_4097", kind="ell_grid", op="product", side=4097, dtype="float64"),
        # the residual of the same form at an ordinary size, in the inner precision of a mixed solver
        dict(name="ell_defect_513_f32", kind="ell_grid", op="defect", side=513, dtype="float32"),
        # an unstructured banded matrix: 5 to 13 entries a row within 2048 columns of the diagonal, rows odd
        dict(name="ell_scatter_4m", kind="ell_scatter", op="product", rows=4194301, half=2048, low=5, high=13,
             dtype="float64"),
        # the smallest call: one smoother sweep on a coarse grid, as a host-driven cycle makes many of
        dict(name="q1_sweep_129", kind="q1", op="jacobi", side=129, dtype="float32"),
        # plain conjugate gradients on the banded Poisson matrix of 66,049 unknowns, to 1e-8
        dict(name="cg_q1_257", kind="cg", form="q1", side=257, tol=1e-8),
        # Jacobi-preconditioned conjugate gradients on an ELL diffusion matrix with jumping coefficients
        dict(name="pcg_ell_513", kind="pcg", level=9, tol=1e-8),
        # the same system for 64 right-hand sides at once
        dict(name="pcg_multi_513", kind="pcg_multi", level=9, columns=64, tol=1e-8),
        # one mixed-precision multigrid solve to 1e-8: a small grid, an ordinary one and the largest
        dict(name="mg_129", kind="mg", level=7, tol=1e-8),
        dict(name="mg_1025", kind="mg", level=10, tol=1e-8),
        dict(name="mg_4097", kind="mg", level=12, tol=1e-8),
        # 64 right-hand sides of the diffusion problem in one multigrid batch
        dict(name="mg_batch_513", kind="mg_batch", level=9, slots=64, tol=1e-8),
        # a burst of requests of mixed sizes at the server, each with a right-hand side of its own
        dict(name="serve_48", kind="serve", requests=48, top=11),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _tolerance(rng, low, high):
    return float("%.2g" % 10.0 ** rng.uniform(math.log10(low), math.log10(high)))


def draw(rng):
    kind = rng.choice(["ell_grid", "ell_grid", "ell_scatter", "q1", "cg", "cg", "pcg", "pcg_multi", "mg", "mg",
                       "mg_batch", "serve"])
    if kind == "ell_grid":
        return dict(kind=kind, op=rng.choice(["product", "defect", "jacobi"]), side=_log_int(rng, 129, 2049),
                    dtype=rng.choice(["float64", "float32"]))
    if kind == "ell_scatter":
        low = rng.randint(1, 8)
        return dict(kind=kind, op=rng.choice(["product", "defect"]), rows=_log_int(rng, 1 << 13, 1 << 22),
                    half=_log_int(rng, 64, 2048), low=low, high=rng.randint(low, 16),
                    dtype=rng.choice(["float64", "float32"]))
    if kind == "q1":
        return dict(kind=kind, op=rng.choice(["product", "defect", "jacobi"]), side=_log_int(rng, 129, 2049),
                    dtype=rng.choice(["float64", "float32"]))
    if kind == "cg":
        return dict(kind=kind, form=rng.choice(["q1", "ell"]), side=_log_int(rng, 33, 513),
                    tol=_tolerance(rng, 1e-9, 1e-6))
    if kind == "pcg":
        return dict(kind=kind, level=rng.randint(6, 9), tol=_tolerance(rng, 1e-9, 1e-6))
    if kind == "pcg_multi":
        return dict(kind=kind, level=rng.randint(6, 9), columns=rng.randint(2, 64),
                    tol=_tolerance(rng, 1e-8, 1e-6))
    if kind == "mg":
        return dict(kind=kind, level=rng.randint(6, 11), tol=_tolerance(rng, 1e-10, 1e-7))
    if kind == "mg_batch":
        return dict(kind=kind, level=rng.randint(6, 9), slots=rng.randint(2, 64),
                    tol=_tolerance(rng, 1e-8, 1e-6))
    return dict(kind=kind, requests=rng.randint(6, 48), top=rng.randint(8, 11))


# ------------------------------------------------------------------ inputs
class Vector(hip.DeviceVector):
    """A torch tensor on the GPU as a vector of honei_amd (shared memory)."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.dtype = np.dtype(np.float64 if tensor.dtype == torch.float64 else np.float32)
        self.size = tensor.numel()

    @property
    def ptr(self):
        return self.tensor.data_ptr()


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(g, shape, low, high, dtype=torch.float64):
    return torch.empty(shape, dtype=torch.float64, device="cuda").uniform_(low, high, generator=g).to(dtype)


def _border(side):
    m = torch.zeros((side, side), dtype=torch.bool, device="cuda")
    m[0], m[-1], m[:, 0], m[:, -1] = True, True, True, True
    return m.reshape(-1)


def _offsets(side):
    return [-side - 1, -side, -side + 1, -1, 0, 1, side - 1, side, side + 1]


def _stencil_bands(g, side, dtype):
    """The 9-point Poisson stencil (identity rows on the border) with every coefficient scaled by U[0.5, 1.5],
    made diagonally dominant; a (9, n) tensor, bands in ascending column order."""
    n, border = side * side, _border(side)
    b = _uniform(g, (9, n), 0.5, 1.5)
    b *= -1.0 / 3.0
    b[4] *= -8.0
    b.masked_fill_(border, 0.0)
    b[4] += b.abs().sum(0) - b[4].abs()
    b[4][border] = 1.0
    return b.to(dtype)


def _poisson_bands(side, dtype=torch.float64):
    n, border = side * side, _border(side)
    b = torch.full((9, n), -1.0 / 3.0, dtype=torch.float64, device="cuda")
    b[4] = 8.0 / 3.0
    b.masked_fill_(border, 0.0)
    b[4][border] = 1.0
    return b.to(dtype)


def _diffusion_bands(k, level):
    """Q1 elements of -div(k grad u) on the side 2^level + 1 grid, k constant on TILES x TILES tiles (averaged
    over a cell where it covers several); u = 0 left and right (identity rows, columns eliminated)."""
    cells, side = 1 << level, (1 << level) + 1
    if cells >= TILES:
        c = k.repeat_interleave(cells // TILES, 0).repeat_interleave(cells // TILES, 1)
    else:
        f = TILES // cells
        c = k.reshape(cells, f, cells, f).mean(dim=(1, 3))
    p = torch.zeros((side + 1, side + 1), dtype=torch.float64, device="cuda")
    p[1:-1, 1:-1] = c
    sw, se, nw, ne = p[:-1, :-1], p[:-1, 1:], p[1:, :-1], p[1:, 1:]
    b = torch.stack([-sw / 3, -(sw + se) / 6, -se / 3, -(sw + nw) / 6, (2.0 / 3.0) * (sw + se + nw + ne),
                     -(se + ne) / 6, -nw / 3, -(nw + ne) / 6, -ne / 3])
    fixed = torch.zeros((side, side), dtype=torch.bool, device="cuda")
    fixed[:, 0], fixed[:, -1] = True, True
    b[:, fixed] = 0.0
    for q in (0, 3, 6):
        b[q][:, 1] = 0.0
    for q in (2, 5, 8):
        b[q][:, -2] = 0.0
    b[4][fixed] = 1.0
    return b.reshape(9, -1)


def _tiles(seed):
    return torch.randn((TILES, TILES), dtype=torch.float64, device="cuda", generator=_gen(seed)).exp()


def _diffusion_rhs(seed, level, count):
    side = (1 << level) + 1
    b = _uniform(_gen(seed + 1), (count, side, side), -1.0, 1.0)
    b[:, :, 0], b[:, :, -1] = 0.0, 0.0
    return b.reshape(count, side * side)


def _poisson_rhs(g, side):
    b = _uniform(g, (side * side,), -1.0, 1.0)
    b[_border(side)] = 0.0
    return b


def _ell_of_bands(bands, side):
    """(columns, values, lengths) of the non-zero entries of every row, ascending, as (slots, n) tensors."""
    n = side * side
    cols = torch.arange(n, device="cuda")[None, :] + torch.tensor(_offsets(side), device="cuda")[:, None]
    keep = (bands != 0) & (cols >= 0) & (cols < n)
    slot = keep.cumsum(0) - 1
    length = keep.sum(0)
    k = int(length.max())
    c = torch.zeros((k, n), dtype=torch.int64, device="cuda")
    v = torch.zeros((k, n), dtype=bands.dtype, device="cuda")
    for q in range(9):
        at = keep[q].nonzero().reshape(-1)
        c[slot[q, at], at] = cols[q, at]
        v[slot[q, at], at] = bands[q, at]
    return c, v, length


def _ell_host(c, v, length):
    """The host arrays of a SparseMatrixELL (one lane per row, stride a multiple of 32)."""
    k, n = c.shape
    stride = 32 * ((n + 31) // 32)
    aj, ax = np.zeros((k, stride), np.uint64), np.zeros((k, stride), NUMPY[str(v.dtype)[6:]])
    torch.from_numpy(aj.view(np.int64))[:, :n] = c.cpu()
    torch.from_numpy(ax)[:, :n] = v.cpu()
    return dict(rows=n, cols=n, stride=stride, ncpr=k, threads=1, Aj=aj.reshape(-1), Ax=ax.reshape(-1),
                Arl=length.cpu().numpy().astype(np.uint64))


def _scatter(g, case):
    """Rows of low..high entries: the diagonal and distinct columns within `half` of it, ascending; values
    N(0, 1), the diagonal dominant."""
    n, k = case["rows"], case["high"]
    r = torch.arange(n, device="cuda")
    length = torch.randint(case["low"], k + 1, (n,), generator=g, device="cuda")
    lo = (r - case["half"]).clamp_min(0)
    room = (r + case["half"]).clamp_max(n - 1) - lo
    big = 1 << 40
    u = (torch.rand((k, n), generator=g, device="cuda", dtype=torch.float64) * (room - k + 1)).long()
    off = torch.arange(k, device="cuda")[:, None]
    u = torch.where(off < length - 1, u, big).sort(0).values + off
    c = lo + u
    c = torch.where(c >= r, c + 1, c)
    used = off < length - 1
    v = torch.randn((k, n), generator=g, device="cuda", dtype=torch.float64) * used
    c = torch.where(used, c, big)
    # the diagonal takes the last slot, which no row's other entries use
    c[k - 1], v[k - 1] = r, 1.0 + v.abs().sum(0)
    c, order = c.sort(0)
    v = v.gather(0, order)
    return torch.where(c < big, c, 0), v.to(TORCH[case["dtype"]]), length


def _matrix(case, seed):
    """Of a single product, defect or sweep: the matrix as (columns, values, lengths) or bands, x, rhs, dinv."""
    g, t = _gen(seed), TORCH[case["dtype"]]
    if case["kind"] == "ell_scatter":
        m = _scatter(g, case)
        n, diag = case["rows"], None
    else:
        m = _stencil_bands(g, case["side"], t)
        n, diag = case["side"] ** 2, m[4]
    x = _uniform(g, (n,), -1.0, 1.0, t)
    rhs = _uniform(g, (n,), -1.0, 1.0, t) if case["op"] != "product" else None
    dinv = (0.7 / diag.double()).to(t) if case["op"] == "jacobi" else None
    return m, x, rhs, dinv


def _serve_levels(case):
    """Sides log-uniform on [65, 2^top + 1], each request at the nearest 2^k + 1; the same mix for every seed."""
    r = np.random.default_rng(case["requests"])
    s = np.exp(r.uniform(math.log(65.0), math.log((1 << case["top"]) + 1.0), case["requests"]))
    return [int(v) for v in np.clip(np.rint(np.log2(s - 1.0)), 6, case["top"])]


# --------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("ell_grid", "ell_scatter", "q1"):
        m, x, rhs, dinv = _matrix(case, seed)
        s = dict(kind=kind, op=case["op"], x=Vector(x), y=Vector(torch.empty_like(x)))
        s["rhs"] = Vector(rhs) if rhs is not None else None
        s["dinv"] = Vector(dinv) if dinv is not None else None
        if kind == "q1":
            s["A"] = hip.Q1Matrix(list(m.cpu().numpy()))
        else:
            s["A"] = hip.EllMatrix.from_dict(_ell_host(*(m if kind == "ell_scatter" else
                                                         _ell_of_bands(m, case["side"]))))
        return s
    if kind == "cg":
        side = case["side"]
        b = _poisson_rhs(_gen(seed), side)
        bands = _poisson_bands(side)
        A = (hip.Q1Matrix(list(bands.cpu().numpy())) if case["form"] == "q1" else
             hip.EllMatrix.from_dict(_ell_host(*_ell_of_bands(bands, side))))
        return dict(kind=kind, form=case["form"], A=A, b=Vector(b), x=Vector(torch.zeros_like(b)),
                    tol=case["tol"])
    if kind in ("pcg", "pcg_multi"):
        level = case["level"]
        bands = _diffusion_bands(_tiles(seed), level)
        A = hip.EllMatrix.from_dict(_ell_host(*_ell_of_bands(bands, (1 << level) + 1)))
        columns = case.get("columns", 1)
        b = _diffusion_rhs(seed, level, columns).T.contiguous()
        return dict(kind=kind, A=A, P=Vector(1.0 / bands[4]), b=Vector(b), x=Vector(torch.zeros_like(b)),
                    columns=columns, tol=case["tol"])
    if kind == "mg":
        b = _poisson_rhs(_gen(seed), (1 << case["level"]) + 1)
        mg = hip.MGSolver(hip.mg_params(MIN_LEVEL, case["level"], tolerance=case["tol"]))
        return dict(kind=kind, mg=mg, b=Vector(b), x=Vector(torch.zeros_like(b)))
    if kind == "mg_batch":
        level, k = case["level"], _tiles(seed)
        host = {}
        for L in range(MIN_LEVEL, level + 1):
            host[L] = _ell_of_bands(_diffusion_bands(k, L), (1 << L) + 1)
        a32 = {L: _ell_host(c, v.float(), n) for L, (c, v, n) in host.items()}
        mg = hip.MGSolver.from_ell(hip.mg_params(MIN_LEVEL, level, tolerance=case["tol"], mask=LEFT_RIGHT),
                                   _ell_host(*host[level]), a32, slots=case["slots"])
        b = _diffusion_rhs(seed, level, case["slots"])
        x = torch.zeros_like(b)
        return dict(kind=kind, mg=mg, b=[Vector(v) for v in b], x=[Vector(v) for v in x], out=x)
    levels, g = _serve_levels(case), _gen(seed)
    server = hip.Server(hip.serve_params(MIN_LEVEL, 6, case["top"]))
    b = [_poisson_rhs(g, (1 << L) + 1) for L in levels]
    return dict(kind=kind, server=server, levels=levels, b=[Vector(v) for v in b],
                x=[Vector(torch.empty_like(v)) for v in b])


def run(state):
    kind = state["kind"]
    if kind == "q1":
        A, x, y = state["A"], state["x"], state["y"]
        if state["op"] == "product":
            hip.q1_product(A, x, y)
        elif state["op"] == "defect":
            hip.q1_defect(A, state["rhs"], x, y)
        else:
            hip.q1_jacobi(A, state["rhs"], state["dinv"], x, y)
        return y.tensor
    if kind in ("ell_grid", "ell_scatter"):
        if state["op"] == "jacobi":
            state["A"].jacobi(state["rhs"], state["dinv"], state["x"], state["y"])
        else:
            state["A"].spmv(state["x"], state["y"], rhs=state["rhs"])
        return state["y"].tensor
    if kind == "serve":
        server = state["server"]
        ids = [server.submit(L, b=b, x=x) for L, b, x in zip(state["levels"], state["b"], state["x"])]
        got = server.drain(len(ids))
        return [x.tensor for x in state["x"]], np.array([got[i]["outer"] for i in ids])
    if kind == "mg_batch":
        for x in state["x"]:
            x.fill(0.0)
        infos = state["mg"].solve_batch(state["b"], state["x"])
        return state["out"], np.array([(i["outer"], i["inner"]) for i in infos])
    b, x = state["b"], state["x"]
    x.fill(0.0)
    if kind == "mg":
        info = state["mg"].solve(b, x)
        return x.tensor, info["outer"], info["inner"]
    if kind == "cg":
        used, _ = (hip.cg_q1 if state["form"] == "q1" else hip.cg_ell)(state["A"], b, x, eps=state["tol"])
        return x.tensor, used
    if kind == "pcg":
        used, _ = hip.pcg_jac_ell(state["A"], state["P"], b, x, eps=state["tol"])
        return x.tensor, used
    used, _ = hip.cg_ell_multi(state["A"], state["P"], b, x, state["columns"], eps=state["tol"])
    return x.tensor, used.astype(np.int64)


# ------------------------------------------------------------ work and exact
def work(case):
    """Of an iterative solve: the iterations that it takes (as measured, to a factor near one), each with its
    matrix read once and every vector that it has to read or write moved once; a multigrid cycle smooths down
    and up (each reads x, rhs or defect and writes x and the next right-hand side or defect) with the matrix at
    a byte a node where it is the constant-coefficient one, 40 bytes otherwise, shared by a batch."""
    kind = case["kind"]
    s = 8 if case.get("dtype", "float64") == "float64" else 4
    if kind in ("ell_grid", "ell_scatter", "q1"):
        n = case["rows"] if kind == "ell_scatter" else case["side"] ** 2
        per = (case["low"] + case["high"]) / 2 if kind == "ell_scatter" else 9
        vectors = {"product": 2, "defect": 3, "jacobi": 4}[case["op"]]
        index = 2 * per + 1 if kind == "ell_scatter" else 0
        return {"bytes": n * (per * s + index + vectors * s), "flops": n * (2 * per + vectors - 2)}
    if kind == "cg":
        n = case["side"] ** 2
        iterations = 2.04 * case["side"]
        return {"bytes": iterations * n * (72 + 72), "flops": iterations * n * 27}
    if kind in ("pcg", "pcg_multi"):
        n, r = ((1 << case["level"]) + 1) ** 2, case.get("columns", 1)
        iterations = 3.8 * (1 << case["level"])
        return {"bytes": iterations * n * (80 + 72 * r), "flops": iterations * n * 31 * r}
    if kind == "serve":
        sizes = [((1 << L) + 1) ** 2 for L in _serve_levels(case)]
        slots, matrix, matrix64, cycles = sum(sizes), 1, 1, 12
        n = 1
    else:
        n = ((1 << case["level"]) + 1) ** 2
        slots = n * case.get("slots", 1)
        matrix, matrix64, cycles = (1, 1, 12) if kind == "mg" else (40, 72, 46)
        if kind == "mg_batch":
            matrix, matrix64 = matrix / case["slots"], matrix64 / case["slots"]
    cycle = slots * 4 / 3 * (2 * 17 + 2 * matrix)
    outer = slots * (28 + 20 + 12 + matrix64)
    return {"bytes": cycles * cycle + cycles / 2 * outer, "flops": slots * (cycles * 4 / 3 * 110 + cycles / 2 * 25)}


def _poisson_exact(b, side):
    """The solution of the 9-point Poisson system: the interior operator is diagonal in the sine basis."""
    m = side - 2
    j = torch.arange(1, m + 1, dtype=torch.float64, device="cuda")
    phase = (j[:, None] * j[None, :]) % (2 * (m + 1))
    sine = torch.sin(phase * (math.pi / (m + 1)))
    c = torch.cos(j * (math.pi / (m + 1)))
    eigen = 8.0 / 3.0 - (2 * c[:, None] + 2 * c[None, :] + 4 * c[:, None] * c[None, :]) / 3.0
    f = b.reshape(side, side)[1:-1, 1:-1].contiguous()
    u = sine @ (((sine @ f @ sine) / eigen) @ sine) * (2.0 / (m + 1)) ** 2
    x = torch.zeros((side, side), dtype=torch.float64, device="cuda")
    x[1:-1, 1:-1] = u
    return x.reshape(-1)


def _diffusion_exact(bands, side, b):
    """Jacobi-preconditioned CG in 64 bits on the columns of b (n, r), well past the tolerance of a solve."""
    n, pad = side * side, side + 1
    inv = (1.0 / bands[4])[:, None]

    def product(p):
        q = torch.nn.functional.pad(p, (0, 0, pad, pad))
        y = bands[4][:, None] * p
        for k, o in enumerate(_offsets(side)):
            if k != 4:
                y.addcmul_(bands[k][:, None], q[pad + o:pad + o + n])
        return y

    x = torch.zeros_like(b)
    r = b.clone()
    p = inv * r
    rz = (r * p).sum(0)
    first = r.square().sum(0)
    for i in range(20 * side):
        v = product(p)
        a = rz / (p * v).sum(0).clamp_min(1e-300)
        x += a * p
        r -= a * v
        z = inv * r
        new = (r * z).sum(0)
        p = z + (new / rz.clamp_min(1e-300)) * p
        rz = new
        if i % 50 == 49 and bool((r.square().sum(0) <= 1e-24 * first).all()):
            break
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind in ("ell_grid", "ell_scatter", "q1"):
        m, x, rhs, dinv = _matrix(case, seed)
        xd = x.double()
        y = torch.zeros_like(xd)
        if kind == "ell_scatter":
            for c, v in zip(m[0], m[1]):
                y += v.double() * xd[c]
        else:
            n = x.numel()
            pad = case["side"] + 1
            xp = torch.nn.functional.pad(xd, (pad, pad))
            for k, o in enumerate(_offsets(case["side"])):
                y += m[k].double() * xp[pad + o:pad + o + n]
        if case["op"] == "product":
            return y
        d = rhs.double() - y
        return d if case["op"] == "defect" else xd + d * dinv.double()
    if kind == "cg":
        return _poisson_exact(_poisson_rhs(_gen(seed), case["side"]), case["side"]), None
    if kind == "mg":
        side = (1 << case["level"]) + 1
        return _poisson_exact(_poisson_rhs(_gen(seed), side), side), None, None
    if kind == "serve":
        g = _gen(seed)
        return [_poisson_exact(_poisson_rhs(g, (1 << L) + 1), (1 << L) + 1) for L in _serve_levels(case)], None
    level, side = case["level"], (1 << case["level"]) + 1
    bands = _diffusion_bands(_tiles(seed), level)
    b = _diffusion_rhs(seed, level, case.get("columns", case.get("slots", 1)))
    x = _diffusion_exact(bands, side, b.T.contiguous())
    if kind == "mg_batch":
        return x.T.contiguous(), None
    return (x.reshape(-1) if kind == "pcg" else x), None
