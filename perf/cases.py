"""What this library's speed is measured on: the calls its users make, from the
smallest solve to the largest batch.

A case is one call on an operator that is already resident in HBM: the setup
(partition, ILUT, low-rank corrections) and the upload are done once per
operator and serve every right-hand side that follows, as a program does that
keeps an operator.  New inputs are new right-hand sides.

Kinds of call:
  solve  Workspace.fgmres from a zero initial guess to 1e-8
  apply  Workspace.apply, one application of the preconditioner (the
         hypre-style use: the caller owns the Krylov loop)
  spmv   Workspace.spmv, y = alpha A x
  serve  Server.submit / Server.wait, several requests in host memory

Problems are the repository's own configurations (bench.py, tests/problems.py):
5- and 7-point Laplacians, upwind convection-diffusion with coefficient 0.3 and
the complex-shifted Laplacian, right-hand sides b = A x* with x* ~ U[-1, 1].
"""
import collections

import numpy as np
import torch

import pargemslr_amd as pg

SHIFT = 0.2 + 0.02j  # the complex-shifted Laplacian of the serving configuration
CONV = 0.3           # coefficient of the convection-diffusion operator
ORTH = {"mgs": pg.PGS_ORTH_MGS, "cgs2": pg.PGS_ORTH_CGS2, "dcgs2": pg.PGS_ORTH_DCGS2}
SERVE_COLUMNS = (1, 3, 8, 2, 5, 16)  # requests of 1 to 16 columns, as the serving stream sends them


def case(kind, family, nx, ny, nz, nrhs, prec="fp64", orth="dcgs2", nlev=3, ncomp=64, droptol=1e-3, fill=20, rank=16,
         kdim=50, name=None):
    c = dict(kind=kind, family=family, nx=nx, ny=ny, nz=nz, nrhs=nrhs, prec=prec, orth=orth, nlev=nlev, ncomp=ncomp,
             droptol=droptol, fill=fill, rank=rank, kdim=kdim)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the quick-start and smoke solve: a small 2D problem, where launches and latency are all there is
        case("solve", "laplacian", 64, 64, 1, 1, nlev=2, ncomp=4, droptol=1e-2, fill=10, rank=0, kdim=30,
             name="solve 64x64 fp64"),
        # the C++ surface's default method (modified Gram-Schmidt, as the reference's), one right-hand side
        case("solve", "laplacian", 48, 48, 48, 1, orth="mgs", name="solve 48^3 fp64 mgs"),
        # the Python call with its defaults (FP64, CGS2) on an odd-sized nonsymmetric grid, a few columns
        case("solve", "convdiff", 41, 37, 29, 4, orth="cgs2", ncomp=8, name="solve cd 41x37x29 fp64 x4 cgs2"),
        # a complex (Helmholtz-like) operator, complex64 apply in complex128 FGMRES, a small batch
        case("solve", "shifted", 32, 32, 32, 4, prec="fp32", ncomp=8, name="solve shifted 32^3 mixed x4"),
        # a served batch: convection-diffusion, as many columns as a server batch takes
        case("solve", "convdiff", 96, 96, 96, 16, prec="fp32", name="solve cd 96^3 mixed x16"),
        # one large solve alone, the mixed form (latency of a single request)
        case("solve", "laplacian", 128, 128, 128, 1, prec="fp32", name="solve 128^3 mixed"),
        # the benchmark's throughput batch
        case("solve", "laplacian", 128, 128, 128, 64, prec="fp32", name="solve 128^3 mixed x64"),
        # the request loop: six requests of 1 to 16 columns handed over and returned in host memory
        case("serve", "laplacian", 64, 64, 64, sum(SERVE_COLUMNS), prec="fp32", name="serve 64^3 mixed"),
        # the preconditioner alone, called from somebody else's Krylov loop, one large vector
        case("apply", "laplacian", 128, 128, 128, 1, name="apply 128^3 fp64"),
        # the same for a few columns of a large 2D problem of odd size
        case("apply", "laplacian", 1023, 1021, 1, 8, name="apply 1023x1021 fp64 x8"),
        # the matrix product alone: one vector, and a block of columns
        case("spmv", "laplacian", 128, 128, 128, 1, name="spmv 128^3 fp64"),
        case("spmv", "laplacian", 1023, 1021, 1, 32, name="spmv 1023x1021 fp64 x32"),
    ]


def draw(rng):
    """A case of the same kinds and ranges.  Two-dimensional and complex grids
    stay at the sizes where restarted FGMRES converges in a few cycles."""
    def size(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["solve", "solve", "solve", "apply", "spmv"])
    family = rng.choice(["laplacian", "laplacian", "plane", "convdiff", "shifted"])
    prec = rng.choice(["fp64", "fp32", "fp32"]) if kind == "solve" else "fp64"
    orth = rng.choice(["dcgs2", "dcgs2", "cgs2", "mgs"])
    if family == "plane":
        family, nx, ny, nz = "laplacian", size(48, 700), size(48, 700), 1
        prec = "fp64"
    elif family == "shifted":
        nx, ny, nz = size(12, 36), size(12, 36), size(12, 36)
    else:
        nx, ny, nz = size(16, 112), size(16, 112), size(16, 112)
    n = nx * ny * nz
    nrhs = 1 << rng.randrange(0, 5 if family == "shifted" else 7)
    while n * nrhs > (1 << 26):
        nrhs //= 2
    ncomp = 4 if n < 8000 else 8 if n < 60000 else 16 if n < 200000 else 64
    return case(kind, family, nx, ny, nz, nrhs, prec=prec, orth=orth, nlev=2 if n < 8000 else 3, ncomp=ncomp,
                kdim=rng.choice([30, 50, 50]))


# ------------------------------------------------------------------ operators
_ops = collections.OrderedDict()  # resident operators, the last few
_ws = collections.OrderedDict()   # the workspace (or server) of the last one


def _kept(cache, key, make, most):
    if key in cache:
        cache.move_to_end(key)
    else:
        while len(cache) >= most:
            cache.popitem(last=False)
        cache[key] = make()
    return cache[key]


def _operator(c):
    grid = (c["nx"], c["ny"], c["nz"])
    key = (c["family"],) + grid + (c["nlev"], c["ncomp"], c["droptol"], c["fill"], c["rank"])

    def make():
        if c["family"] == "convdiff":
            A = pg.convdiff(*grid, CONV)
        elif c["family"] == "shifted":
            A = pg.laplacian(*grid, shift=SHIFT, complex_=True)
        else:
            A = pg.laplacian(*grid)
        return pg.DevOp(pg.Gemslr(A, pg.config_params(c["nlev"], c["ncomp"], c["droptol"], c["fill"], c["rank"])))

    return key, _kept(_ops, key, make, 3)


def _stencil(c, x, scale=1.0):
    """scale * A x for x of shape (n, nrhs), from the grid's stencil."""
    shape = (c["nz"], c["ny"], c["nx"], x.shape[1])
    v = x.view(shape)
    ones = sum(d == 1 for d in shape[:3])
    if c["family"] == "convdiff":
        diag, up, down = 6.0 + 3.0 * CONV, -1.0 - CONV, -1.0
    else:
        diag, up, down = (4.0 if ones else 6.0) - (SHIFT if c["family"] == "shifted" else 0.0), -1.0, -1.0
    y = v * (scale * diag)
    for d in range(3):
        m = shape[d] - 1
        if m > 0:
            y.narrow(d, 1, m).add_(v.narrow(d, 0, m), alpha=scale * up)
            y.narrow(d, 0, m).add_(v.narrow(d, 1, m), alpha=scale * down)
    return y.view(x.shape)


def _uniform(c, seed):
    """Values in [-1, 1] (both parts of a complex one), n x nrhs on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    shape = (c["nx"] * c["ny"] * c["nz"], c["nrhs"])
    if c["family"] == "shifted":
        t = torch.rand(shape + (2,), generator=g, device="cuda", dtype=torch.float64)
        return torch.view_as_complex(t.mul_(2.0).sub_(1.0))
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float64).mul_(2.0).sub_(1.0)


ALPHA = 1.5  # of y = alpha A x


def prepare(case, seed):
    c = case
    key, D = _operator(c)
    s = {"case": c, "prec": pg.PGS_PREC_FP64 if c["prec"] == "fp64" else pg.PGS_PREC_FP32}
    if c["kind"] == "serve":
        def serve():
            S = pg.Server(max_batch=16, kdim=c["kdim"], prec=s["prec"], orth=ORTH[c["orth"]])
            return S, S.add_operator(D)

        s["server"], s["op"] = _kept(_ws, key + ("serve",), serve, 1)
        b = _stencil(c, _uniform(c, seed)).cpu().numpy()
        at = np.cumsum((0,) + SERVE_COLUMNS)
        s["b"] = [np.ascontiguousarray(b[:, at[i]:at[i + 1]]) for i in range(len(SERVE_COLUMNS))]
        return s
    kdim = c["kdim"] if c["kind"] == "solve" else 1
    s["ws"] = _kept(_ws, key + (c["nrhs"], kdim), lambda: pg.Workspace(D, max_nrhs=c["nrhs"], kdim=kdim), 1)
    x = _uniform(c, seed)
    if c["kind"] == "solve":
        s["b"] = _stencil(c, x)
        s["x"] = torch.empty_like(x)
    elif c["kind"] == "apply":
        s["v"] = x
        s["z"] = torch.empty_like(x)
    else:
        s["x"] = x
        s["y"] = torch.empty_like(x)
    return s


def run(state):
    s = state
    c = s["case"]
    if c["kind"] == "solve":
        s["x"].zero_()
        r = s["ws"].fgmres(s["b"], s["x"], nrhs=c["nrhs"], kdim=c["kdim"], tol=1e-8, prec=s["prec"], orth=ORTH[c["orth"]])
        return {"x": s["x"], "iters": np.array([q[1] for q in r], dtype=np.int64)}
    if c["kind"] == "apply":
        s["ws"].apply(s["v"], s["z"], nrhs=c["nrhs"], prec=s["prec"])
        return s["z"]
    if c["kind"] == "spmv":
        s["ws"].spmv(s["x"], s["y"], alpha=ALPHA, nrhs=c["nrhs"])
        return s["y"]
    reqs = [s["server"].submit(s["op"], b) for b in s["b"]]
    return [s["server"].wait(r)[0] for r in reqs]


def exact(case, seed):
    """Solves: the x* that b was made from.  Products: the stencil.  The
    preconditioner has no value apart from this library's own factors."""
    c = case
    if c["kind"] == "apply":
        return None
    x = _uniform(c, seed)
    if c["kind"] == "solve":
        return {"x": x, "iters": None}
    if c["kind"] == "spmv":
        return _stencil(c, x, ALPHA)
    h = x.cpu().numpy()
    at = np.cumsum((0,) + SERVE_COLUMNS)
    return [np.ascontiguousarray(h[:, at[i]:at[i + 1]]) for i in range(len(SERVE_COLUMNS))]


def work(case):
    """The operator's arrays, the inputs and the outputs, once each: what any
    method has to touch.  A solve reads the operator once per iteration, and
    the iterations are not known before it runs, so its figure is a floor of
    one iteration.  The factors hold about 37 entries per row for a 7-point
    grid with fill 20 and about 20 for a 5-point one, at most twice the fill."""
    c = case
    n = c["nx"] * c["ny"] * c["nz"]
    flat = c["nz"] == 1
    cx = 2 if c["family"] == "shifted" else 1
    full = 8 * cx
    low = full if c["prec"] == "fp64" else full // 2
    nnz = n * (5 if flat else 7)
    factors = n * min(20 if flat else 37, 2 * c["fill"])
    block = n * c["nrhs"] * full
    mat = nnz * (full + 4) + 4 * (n + 1)
    pre = factors * (low + 4)
    mul = 2 * c["nrhs"] * cx * cx
    if c["kind"] == "spmv":
        return {"bytes": mat + 2 * block, "flops": nnz * mul}
    if c["kind"] == "apply":
        return {"bytes": pre + 2 * block, "flops": 2 * factors * mul}
    return {"bytes": mat + pre + 2 * block, "flops": (nnz + 2 * factors) * mul}
