"""The ring solve's waves (solving, copying records, copying row data) at the
sizes where their hand-over can go wrong: blocks of fewer steps than stages, step
counts around a multiple of the stages, half and whole steps, every number of
columns per workgroup, and rings so large that fewer stages fit in LDS.

Bounds: the apply within 1e-12 (FP64), 1e-5 (FP32) and 1e-4 (complex64) of the
oracle, as the other kernels; repeated applies give the same bits (a stage that
is read too early or overwritten too soon does not)."""
import numpy as np
import pytest

import pargemslr_amd as pg
from tests import problems as P

pytestmark = pytest.mark.gpu

GRIDS = {"5x4x3": ((5, 4, 3), 2, 2), "9x1x1": ((9, 1, 1), 1, 1), "13x11x7": ((13, 11, 7), 3, 4),
         "33x31": ((33, 31, 1), 2, 4), "17x16x15": ((17, 16, 15), 2, 4)}


def _check(A, G, columns, gpu):
    O = P.oracle_of(G)
    D = pg.DevOp(G, device=gpu)
    cx = A.is_complex
    for nr in columns:
        W = pg.Workspace(D, max_nrhs=nr, kdim=1)
        V = np.stack([(pg.rng_normal(7 + c, 2 * A.n).view(np.complex128) if cx else pg.rng_normal(7 + c, A.n))
                      for c in range(nr)], axis=1)
        ref = np.stack([O.apply(V[:, c]) for c in range(nr)], axis=1)
        v = pg.DeviceArray.from_numpy(np.ascontiguousarray(V), device=gpu)
        for prec, tol in ((pg.PGS_PREC_FP64, 1e-12), (pg.PGS_PREC_FP32, 1e-4 if cx else 1e-5)):
            first = None
            for _ in range(4):
                z = pg.DeviceArray(V.shape, dtype=V.dtype, device=gpu)
                W.apply(v, z, nrhs=nr, prec=prec)
                pg.synchronize(gpu)
                Z = z.numpy()
                first = Z if first is None else first
                assert np.array_equal(Z, first), (nr, prec)
            err = np.linalg.norm(first - ref, axis=0) / np.linalg.norm(ref, axis=0)
            assert err.max() <= tol, (nr, prec, err.max())
        W.close()
    D.close()


@pytest.mark.parametrize("geom", ["", "64x4", "128x4"])
@pytest.mark.parametrize("cols", ["", "1", "2", "4", "8", "16"])
def test_columns_and_steps(geom, cols, gpu, monkeypatch):
    """Half and whole steps, each number of columns per workgroup forced (a
    smaller number where LDS or the batch holds no more), 1 to 64 columns."""
    if geom:
        monkeypatch.setenv("PGS_RING_GEOM", geom)
    if cols:
        monkeypatch.setenv("PGS_TRSV_CG", cols)
    for name in ("13x11x7", "33x31"):
        grid, nlev, ncomp = GRIDS[name]
        A = pg.laplacian(*grid)
        _check(A, P.setup(A, nlev, ncomp, 1e-3, 20, 4), (1, 4, 64), gpu)


@pytest.mark.parametrize("name", sorted(GRIDS))
@pytest.mark.parametrize("geom", ["64x4", "128x4"])
def test_small_blocks(name, geom, gpu, monkeypatch):
    monkeypatch.setenv("PGS_RING_GEOM", geom)
    grid, nlev, ncomp = GRIDS[name]
    for A in (pg.convdiff(*grid, 0.3), pg.laplacian(*grid, shift=0.2 + 0.02j, complex_=True)):
        _check(A, P.setup(A, nlev, ncomp, 1e-3, 20, 0), (1, 2, 8), gpu)


@pytest.mark.parametrize("rows,cx", [(15000, False), (7500, True)], ids=["fp64-4-stages", "complex128-2-stages"])
def test_large_rings(rows, cx, gpu):
    """Row rows + i depends on row i alone: two level sets and a window of
    `rows`, so that a ring of one column leaves LDS for few stages."""
    n = 2 * rows
    import scipy.sparse as sp
    d = np.full(n, 4.0 + (0.5j if cx else 0.0))
    o = -1.0 - pg.rng_uniform(3, rows, 0.0, 0.5)
    M = sp.csr_matrix(sp.diags([d, o], [0, -rows]))
    A = P.csr_from_scipy(M)
    _check(A, P.setup(A, 1, 1, 1e-6, 20, 0, perm=0), (1, 2), gpu)
