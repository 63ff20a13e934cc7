"""Wide batches of few rows, where the delayed-CGS2 dots and the MGS sweeps take
more workgroups than one per 256 rows: as many as the partials' buffer holds, or
as the pieces ask for, with their sums in the next kernel or in a launch of their
own.

Steps, oracle and bounds as in the test of the kernels that close a step."""
import pytest

import pargemslr_amd as pg
from tests.test_gpu_krylov_steps import ops, test_fixed_steps as fixed_steps  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("orth", [pg.PGS_ORTH_MGS, pg.PGS_ORTH_DCGS2], ids=["mgs", "dcgs2"])
@pytest.mark.parametrize("kdim,maxits", [(7, 17), (40, 40)])
@pytest.mark.parametrize("grid,cx,nr", [((10, 10, 10), True, 64), ((16, 16, 17), True, 32), ((24, 24, 24), True, 64),
                                        ((24, 24, 23), False, 64), ((24, 24, 24), False, 32)])
def test_wide_batches(ops, gpu, grid, cx, nr, kdim, maxits, orth):  # noqa: F811
    fixed_steps(ops, gpu, grid, cx, nr, kdim, maxits, orth)
