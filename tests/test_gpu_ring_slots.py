"""Level solves whose sweep window is shorter than a step: the last row (of L, or
the first one of U) reads rows of the one step before it, which holds 32 rows.
The ring holds a slot for each row of a step; with fewer, rows that nobody reads
share the slots of the rows that are read.

Bounds: the apply within 1e-12 (FP64) and 1e-5 (FP32) of the oracle, as the other
kernels: a 33-row block with pivots 4 and entries of at most 5, far below them."""
import numpy as np
import pytest
import scipy.sparse as sp

import pargemslr_amd as pg
from tests import problems as P

pytestmark = pytest.mark.gpu


def _matrix(cols, upper):
    M = sp.lil_matrix((33, 33))
    M.setdiag(4.0)
    for c in cols:
        if upper:
            M[0, c + 1] = -1.0 - 0.1 * c
        else:
            M[32, c] = -1.0 - 0.1 * c
    return P.csr_from_scipy(sp.csr_matrix(M))


@pytest.mark.parametrize("geom", ["", "64x4", "128x4"])
@pytest.mark.parametrize("cols", [(31,), (28, 31), (18, 31), (17, 31), (16, 31), (13, 31), (2, 31)],
                         ids=lambda c: f"window{33 - c[0]}")
@pytest.mark.parametrize("upper", [False, True], ids=["L", "U"])
def test_window_shorter_than_step(cols, upper, geom, gpu, monkeypatch):
    if geom:
        monkeypatch.setenv("PGS_RING_GEOM", geom)
    A = _matrix(cols, upper)
    G = P.setup(A, 1, 1, 1e-6, 20, 0, perm=0)
    O = P.oracle_of(G)
    D = pg.DevOp(G, device=gpu)
    for nr in (1, 2, 4, 8, 16):
        W = pg.Workspace(D, max_nrhs=nr, kdim=1)
        V = np.stack([pg.rng_normal(7 + c, A.n) for c in range(nr)], axis=1)
        ref = np.stack([O.apply(V[:, c]) for c in range(nr)], axis=1)
        v = pg.DeviceArray.from_numpy(np.ascontiguousarray(V), device=gpu)
        for prec, tol in ((pg.PGS_PREC_FP64, 1e-12), (pg.PGS_PREC_FP32, 1e-5)):
            z = pg.DeviceArray(V.shape, device=gpu)
            W.apply(v, z, nrhs=nr, prec=prec)
            pg.synchronize(gpu)
            err = np.linalg.norm(z.numpy() - ref, axis=0) / np.linalg.norm(ref, axis=0)
            assert err.max() <= tol, (nr, prec, err.max())
        W.close()
    D.close()
