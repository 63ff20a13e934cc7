"""The low-rank term whose update sums stage 1's partials itself: ranks below
and above the 32 of the register kernel, one and several output groups per
workgroup, and batches past the 4096 partials, where a launch of its own does.

Bounds: the apply within 1e-12 (FP64), 1e-5 (FP32) and 1e-4 (complex64) of the
oracle, as the other kernels."""
import numpy as np
import pytest

import pargemslr_amd as pg
from tests import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("rank", [3, 16, 20, 40])
def test_lowrank_term(rank, cx, gpu):
    A = pg.laplacian(17, 16, 15, shift=0.2 + 0.02j, complex_=True) if cx else pg.laplacian(17, 16, 15)
    G = P.setup(A, 3, 4, 1e-3, 20, rank)
    O = P.oracle_of(G)
    D = pg.DevOp(G, device=gpu)
    for nr in (1, 2, 8, 64):
        W = pg.Workspace(D, max_nrhs=nr, kdim=1)
        V = np.stack([(pg.rng_normal(7 + c, 2 * A.n).view(np.complex128) if cx else pg.rng_normal(7 + c, A.n))
                      for c in range(nr)], axis=1)
        ref = np.stack([O.apply(V[:, c]) for c in range(nr)], axis=1)
        v = pg.DeviceArray.from_numpy(np.ascontiguousarray(V), device=gpu)
        for prec, tol in ((pg.PGS_PREC_FP64, 1e-12), (pg.PGS_PREC_FP32, 1e-4 if cx else 1e-5)):
            z = pg.DeviceArray(V.shape, dtype=V.dtype, device=gpu)
            W.apply(v, z, nrhs=nr, prec=prec)
            err = np.linalg.norm(z.numpy() - ref, axis=0) / np.linalg.norm(ref, axis=0)
            assert err.max() <= tol, (nr, prec, err.max())
        W.close()
    D.close()
