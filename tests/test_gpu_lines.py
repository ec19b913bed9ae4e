"""The x-line Green kernel between the separate y and z passes (grids whose
(y, z) planes do not take the fused kernels) against the seven-pass path: new
line lengths, tiles of 16, 8, 4 and 2 columns, column counts that leave the last
tile ragged, odd y and z lengths, FP64 and mixed.  The two paths compute the
same sums in another order, so 40 forced iterations of a contracting loop keep
them within rounding of each other: the bars of the fused-transform test."""
import numpy as np
import pytest

from pyevp import lib

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


@pytest.mark.parametrize("dims", [(12, 10, 9), (36, 50, 27), (60, 7, 5), (100, 12, 10), (144, 5, 6), (160, 9, 7),
                                  (200, 4, 6), (256, 3, 4), (8, 130, 136)])
@pytest.mark.parametrize("prec", [lib.FP64, lib.MIXED])
def test_lines_match_seven_passes(job_factory, dims, prec):
    inp = job_factory(f"lines{dims}", n=0, dims=dims, grains=6, seed=67, increments=1, pore_fraction=0.02,
                      pore_radius=1)
    out = []
    for fused in (True, False):
        job = lib.GpuJob(inp, prec)
        job.set_fused_transforms(fused)
        job.run(1, forced=40)
        out.append((job.state(), job.macro()))
        job.close()
    (A, ma), (B, mb) = out
    tol = 1e-10 if prec == lib.FP64 else 1e-6
    for k in ("Sig", "DisGrad"):
        assert rel(A[k], B[k]) < tol, (k, rel(A[k], B[k]))
    assert rel(A["Edot"], B["Edot"]) < 10 * tol  # the rate goes as sigma^10
    assert rel(ma["sig_avg"], mb["sig_avg"]) < tol


@pytest.mark.parametrize("dims", [(36, 10, 9), (10, 12, 12)])
def test_batches_are_exact_off_the_fused_path(job_factory, dims):
    """Five passes (36 x 10 x 9) and seven (10 x 12 x 12): iterations queued in
    batches, the ones past the loop's end doing nothing, give the state of the
    waiting host bit for bit."""
    inp = job_factory(f"linesb{dims}", n=0, dims=dims, grains=5, seed=71, increments=2, pore_fraction=0.02,
                      pore_radius=1)
    ref = None
    for batch in (0, 1, 3, 4):
        job = lib.GpuJob(inp, lib.MIXED)
        job.set_loop_batch(batch)
        it, _ = job.run(2)
        s = job.state()
        job.close()
        if ref is None:
            ref = (list(it), s)
            continue
        assert list(it) == ref[0], batch
        for k in s:
            assert np.array_equal(s[k], ref[1][k]), (batch, k)
