"""The reverse pass with the last recorded segment's tape still held: the same
gradient, bit for bit, for every checkpoint interval (one segment, several, one
increment each), on a second reverse pass over the same recording (the tape
then holds the first segment) and after other increments were run in between
(the context's state is not what the tape holds)."""
import numpy as np
import pytest

from pyevp import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [lib.FP64, lib.MIXED])
def test_gradient_does_not_depend_on_the_segments(job_factory, prec):
    inp = job_factory("adjtape", n=8, grains=4, seed=73, increments=5, iter_max=60)
    n, ref = 5, None
    seeds = np.random.default_rng(5).standard_normal((n, 6))
    for ck in (5, 2, 1, 4):
        job = lib.GpuJob(inp, prec)
        curve, _ = job.adjoint_record(n, ck)
        g = [job.adjoint_run(seeds, cg_tol=1e-12)[0] for _ in range(2)]
        end = job.state()["Sig"]
        job.run(1)
        g.append(job.adjoint_run(seeds, cg_tol=1e-12)[0])
        assert np.array_equal(job.state()["Sig"], end)  # left in the recorded final state
        job.close()
        if ref is None:
            ref = (curve, g[0])
            assert np.all(np.isfinite(ref[1])) and np.max(np.abs(ref[1])) > 0
        assert np.array_equal(curve, ref[0])
        for x in g:
            assert np.array_equal(x, ref[1]), ck
