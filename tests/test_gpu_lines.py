"""Transforms of the lengths with a Stockham plan that are not multiples of 4,
against numpy (the bars of tests/test_gpu_anysize.py: 1e-12 FP64, 2e-6 FP32),
z lines in groups that do not fill the last workgroup among them; and
the x-line Green kernel between the separate y and z passes (grids whose
(y, z) planes do not take the fused kernels) against the seven-pass path: every
line length, tiles of 16, 8, 4 and 2 columns (4, or 2 at FP64 lengths above 200,
on the small sections; 8 and 16 on those of 512 such tiles and more), column
counts that leave the last tile ragged, odd y and z lengths, FP64 and mixed.
The two paths compute the same sums in another order, so 40 forced iterations
of a contracting loop keep them within rounding of each other: the bars of the
fused-transform test."""
import numpy as np
import pytest

from pyevp import lib

pytestmark = pytest.mark.gpu


# every new length along x or y, every new even one along z; nx ny = 1 or 15 mod 16
@pytest.mark.parametrize("dims", [(15, 25, 10), (27, 45, 18), (75, 3, 30), (125, 5, 50), (225, 3, 54), (5, 15, 90),
                                  (10, 27, 108), (18, 75, 4), (30, 125, 2), (50, 225, 6), (54, 10, 150), (90, 18, 12),
                                  (108, 30, 4), (150, 54, 4), (180, 90, 8), (216, 108, 2), (250, 150, 2), (4, 180, 180),
                                  (3, 216, 216), (3, 250, 250)])
@pytest.mark.parametrize("prec", [lib.FP64, lib.MIXED])
def test_mixed_radix_lengths_vs_numpy(dims, prec):
    rng = np.random.default_rng(sum(dims))
    x = rng.standard_normal(dims)
    tol = 1e-12 if prec == lib.FP64 else 2e-6
    c = lib.Context(*dims, prec)
    X = c.rfftn(x)
    ref = np.fft.rfftn(x)
    assert np.max(np.abs(X - ref)) < tol * np.max(np.abs(ref))
    y = c.irfftn_unnormalised(ref) / x.size
    assert np.max(np.abs(y - x)) < tol * np.max(np.abs(x))
    c.close()


def rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


# every length of the x-line kernel that the grids below do not hold, on sections
# of odd and ragged column counts
SECTIONS = ((3, 5), (5, 4), (7, 3), (2, 9))
LINES = [(nx, *SECTIONS[k % 4]) for k, nx in enumerate(
    (10, 15, 16, 18, 20, 24, 25, 27, 30, 32, 40, 45, 48, 50, 54, 64, 72, 75, 80, 90, 96, 108, 120, 125, 128, 150, 180,
     192, 216, 225, 240, 250))]
GRIDS = [(12, 10, 9), (36, 50, 27), (60, 7, 5), (100, 12, 10), (144, 5, 6), (160, 9, 7), (200, 4, 6), (256, 3, 4),
         (8, 130, 136)] + LINES


# tiles of 16 columns: 8 x 130 x 136 (8970 columns); of 8: the last two (4221)
@pytest.mark.parametrize("prec,dims", [(p, d) for p in (lib.FP64, lib.MIXED) for d in GRIDS] +
                         [(lib.FP64, (36, 67, 125)), (lib.MIXED, (72, 67, 125))])
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


@pytest.mark.parametrize("prec", [lib.MIXED, lib.FP64])
@pytest.mark.parametrize("dims,fused", [((36, 10, 9), True), ((10, 12, 12), True), ((7, 12, 12), True),
                                        ((10, 12, 12), False)])
def test_batches_are_exact_off_the_fused_path(job_factory, dims, fused, prec):
    """Five passes (36 x 10 x 9, 10 x 12 x 12) and seven (7 x 12 x 12, whose nx
    has no x-line kernel, and 10 x 12 x 12 with the fused transforms off):
    iterations queued in batches, the ones past the loop's end doing nothing,
    give the state of the waiting host bit for bit."""
    inp = job_factory(f"linesb{dims}", n=0, dims=dims, grains=5, seed=71, increments=2, pore_fraction=0.02,
                      pore_radius=1)
    ref = None
    for batch in (0, 1, 3, 4):
        job = lib.GpuJob(inp, prec)
        job.set_fused_transforms(fused)
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
