"""The kernels that close a Krylov step (sums of the dots, Hessenberg column and
Givens rotation, norm, back substitution) where their work splits: bases of one
and of several dot chunks, partial sums that the fix adds itself (up to 128
workgroups of dots: 32^3 rows) and that a kernel of their own adds, triangular
systems past 64 vectors, restarts and cycles that end early.

A fixed number of unpreconditioned steps (tol 0) against the oracle's MGS.
Bounds: the operators' condition numbers are below 1e3 and every variant is
backward stable, so iterates and residuals agree to about 1e3 * eps * steps =
2e-11; 1e-9 is asked for."""
import numpy as np
import pytest

import pargemslr_amd as pg
from oracle import oracle as orc
from tests import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(gpu):
    made = {}

    def get(grid, cx):
        if (grid, cx) not in made:
            A = pg.laplacian(*grid, shift=0.1j, complex_=True) if cx else pg.laplacian(*grid)
            made[grid, cx] = (A, pg.DevOp(P.setup(A, 1, 1, 0.5, 2, 0), device=gpu))
        return made[grid, cx]

    yield get
    for _, D in made.values():
        D.close()


@pytest.mark.parametrize("orth", [pg.PGS_ORTH_MGS, pg.PGS_ORTH_CGS2, pg.PGS_ORTH_DCGS2], ids=["mgs", "cgs2", "dcgs2"])
@pytest.mark.parametrize("kdim,maxits", [(1, 3), (7, 17), (17, 17), (64, 50), (100, 70)])
@pytest.mark.parametrize("grid,cx,nr", [((13, 11, 7), False, 1), ((32, 32, 32), False, 1), ((33, 32, 32), False, 1),
                                        ((32, 32, 32), False, 4), ((13, 11, 7), False, 64), ((13, 11, 7), True, 2),
                                        ((13, 11, 7), True, 64)])
def test_fixed_steps(ops, gpu, grid, cx, nr, kdim, maxits, orth):
    A, D = ops(grid, cx)
    rng = np.random.default_rng(5)
    b = rng.standard_normal((A.n, nr))
    if cx:
        b = b + 1j * rng.standard_normal((A.n, nr))
    W = pg.Workspace(D, max_nrhs=nr, kdim=kdim)
    bd = pg.DeviceArray.from_numpy(np.ascontiguousarray(b), device=gpu)
    first = None
    for graph in (False, True):
        xd = pg.DeviceArray.from_numpy(np.zeros_like(b), device=gpu)
        res = W.fgmres(bd, xd, nrhs=nr, kdim=kdim, maxits=maxits, tol=0.0, orth=orth, use_precond=False,
                       use_graph=graph)
        x = xd.numpy()
        first = x if first is None else first
        assert np.array_equal(x, first)
    W.close()
    for c in sorted({0, nr - 1}):
        xo, _, ito, rro, _ = orc.fgmres(A, np.ascontiguousarray(b[:, c]), kdim=kdim, maxits=maxits, tol=0.0)
        assert res[c][1] == ito == maxits
        assert abs(res[c][2] - rro) <= 1e-9 * max(rro, 1e-3)
        assert np.linalg.norm(x[:, c] - xo) <= 1e-9 * np.linalg.norm(xo)


@pytest.mark.parametrize("nr", [16, 32, 64])
def test_mgs_partials(ops, gpu, nr):
    """MGS where every workgroup adds up the dots' partials itself (up to 4096
    values: 16 and 32 columns of 32^3 rows) and where a kernel of its own does."""
    test_fixed_steps(ops, gpu, (32, 32, 32), False, nr, 7, 17, pg.PGS_ORTH_MGS)
