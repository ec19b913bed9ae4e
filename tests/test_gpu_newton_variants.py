"""The loop's Newton kernel in each of its rate-law variants against the
oracle's whole loop: exponents that select the compile-time power (10), the
runtime power of the fast variant (7), the squaring loop (n > 32) and pow()
(12.5, and 0.8 < 1), with equal and unequal forward and backward CRSS, on a
grid that leaves the last wave ragged (630 voxels: 9 waves and 54 lanes) and
mixes gas and crystal voxels in a wave.  Bars: those of the whole-loop parity
tests (rounding, carried through three increments)."""
import pytest

import oracle as O
from pyevp import lib, synth
from test_gpu_parity import _compare_jobs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrs,tau0b", [(10.0, 19.0), (7.0, 16.0), (7.0, 19.0), (33.0, 16.0), (33.0, 19.0),
                                       (12.5, 19.0), (0.8, 16.0)])
def test_newton_variants_vs_oracle(job_factory, nrs, tau0b):
    m = synth.Material(nrs=nrs, tau0b=tau0b)
    inp = job_factory(f"nv{nrs}_{tau0b}", n=0, dims=(10, 9, 7), grains=5, seed=61, increments=3,
                      pore_fraction=0.02, pore_radius=1, material=m)
    _compare_jobs(O.Job(inp), lib.GpuJob(inp), 3)
