"""The phase-field kernels where their LDS runs overflow, bit for bit against
the oracle: lists of up to 10 entries in every voxel (5 per cell on average:
a tile's box holds more entries than the packed lists take, its voxels more
candidate grains than one run of results, and neighbourhoods more grains than
the candidate kernel keeps in registers), on grids with whole tiles and with
ragged ones, down to the smallest."""
import numpy as np
import pytest

import oracle as o
import pf_cases
from pyevp import pf as gpf
from test_gpu_pf import same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4, 8, 8), (8, 16, 16), (9, 10, 11), (5, 9, 17), (3, 3, 3)])
@pytest.mark.parametrize("grains,extra", [(12, 9), (14, 4), (6, 5)])
def test_pf_dense_lists_vs_oracle(shape, grains, extra):
    rng = np.random.default_rng(grains)
    gid = rng.integers(1, grains + 1, shape).astype(np.int32)
    rho = rng.uniform(200.0, 250.0, shape)
    P = pf_cases.params(grains - 2, M_gb=2e-12)
    n, idx, val = pf_cases.random_lists(gid, 7 * grains + extra, cap=o.PF_CAP, extra=extra)
    ra0 = rng.uniform(0, 300, grains + 3)
    r = o.pf_run_lists(n, idx, val, gid, rho, 2, P, ra0)
    pf = gpf.PhaseField(gid.shape, ra0.size)
    try:
        pf.set_lists(n, idx[..., :gpf.CAP], val[..., :gpf.CAP], gid, rho)
        gn, ra = pf.steps(P, 2, ra0)
        same(pf.lists(), r, gn, ra)
    finally:
        pf.close()
