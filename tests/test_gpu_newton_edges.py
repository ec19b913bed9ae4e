"""Inputs at the edge of what the loop's Newton kernel takes: slip systems
switched off by an infinite CRSS (a file or a caller's state may hold one; the
rate is then 0, the reference's division by infinity), in some voxels of a wave
and in one direction only, or in a whole phase, which is then elastic, against
the oracle at the bars of the whole-loop parity tests; and a C0 that is not
positive definite, as a caller may set one."""
import numpy as np
import pytest

import oracle as O
from pyevp import lib, synth

pytestmark = pytest.mark.gpu

FIELDS = (("sig", 6), ("disgrad", 9), ("eps", 6), ("edot", 6), ("tran", 9), ("crss", 24), ("gamacum", 1))


def _download(job):
    s = {k: np.zeros((m, job.n)) for k, m in FIELDS}
    lib._chk(lib.gpu().evpgpu_download_state(job.ctx, *[lib._p(s[k]) for k, _ in FIELDS], None), "download_state")
    return s


def _upload(job, s):
    lib._chk(lib.gpu().evpgpu_upload_state(job.ctx, *[lib._p(np.ascontiguousarray(s[k])) for k, _ in FIELDS]),
             "upload_state")


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def _compare(J, g, increments):
    it_o = J.run(increments)
    it_g, _ = g.run(increments)
    assert list(it_g) == list(it_o)
    s = g.state()
    for k, f in (("Sig", O.SIG), ("Edot", O.EDOT), ("Eps", O.EPS), ("DisGrad", O.DISGRAD), ("TranMat", O.TRANMAT),
                 ("gamdot", O.GAMDOT)):
        assert _rel(s[k], J.field(f)) < 1e-10, k
    c = J.field(O.CRSS)
    off = np.isinf(c)
    assert off.any() and np.array_equal(s["crss"][off], c[off])
    assert _rel(s["crss"][~off], c[~off]) < 1e-10
    g.close()


@pytest.mark.parametrize("nrs,tau0b", [(10.0, 16.0), (10.0, 19.0), (7.0, 16.0), (12.5, 16.0), (12.5, 19.0)])
def test_infinite_crss_switches_a_system_off(job_factory, nrs, tau0b):
    m = synth.Material(nrs=nrs, tau0b=tau0b)
    inp = job_factory(f"inf{nrs}_{tau0b}", n=0, dims=(10, 9, 7), grains=5, seed=61, increments=3, material=m)
    J, g = O.Job(inp), lib.GpuJob(inp)
    both = tau0b == m.tau0f  # else the backward direction alone
    c = J.field(O.CRSS)
    c[::3, 3, 0 if both else 1:] = np.inf
    J.set_field(O.CRSS, c)
    s = _download(g)
    s["crss"] = c.reshape(g.n, 24).T
    _upload(g, s)
    _compare(J, g, 3)


@pytest.mark.parametrize("nrs2", [10.0, 34.0, 12.5])
def test_infinite_crss_of_a_phase(job_factory, nrs2):
    """the elastic phase's exponent only selects the rate law's form"""
    inp = job_factory(f"infphase{nrs2}", n=0, dims=(10, 9, 7), grains=8, seed=7, increments=3,
                      phase2=synth.Material(nrs=nrs2, tau0f=np.inf, tau0b=np.inf))
    _compare(O.Job(inp), lib.GpuJob(inp), 3)


def _loading(job, sign):
    """the job's loading through the caller's entry point, C0 times sign"""
    c066, s066, c0, s0 = job.setup_info()
    ld = lib.Loading(dt=1e-3, err_tol=1e-6, iter_max=2000, update_flag=1, hard_flag=1, elast_bc=1, wgt_ph1=1.0,
                     d_vm0=1.0)
    ld.c066[:], ld.s066[:], ld.c0[:], ld.s0[:] = (sign * c066).ravel(), s066.ravel(), c0.ravel(), s0.ravel()
    ld.velgrad_bc_flag[:], ld.velgrad_bc[:] = (0, 0, 1, 1, 1, 1), (0.0, 0.0, 1.0, 0.0, 0.0, 0.0)
    ld.stress_bc_flag[:] = (1, 1, 0, 0, 0, 0)
    return ld


@pytest.mark.parametrize("shortcut", [True, False])
def test_descent_test_without_bounds_on_c0(job_factory, shortcut):
    """The line search compares |C0 r|^2 of a trial and of its start, and
    bounds from C0's eigenvalues decide most comparisons; a C0 that is not
    positive definite has none, and every comparison is then made.  -C0 is
    such a matrix with the same |C0 r|^2: the same state, bit for bit, and the
    same counts, in a loop that backtracks (the oracle's trace of this one:
    51589 accepted trials, 3150 rejected for their size, 992 backtracks)."""
    inp = job_factory("c0bounds", n=0, dims=(10, 9, 7), grains=5, seed=7, increments=1)
    out = []
    for sign in (1.0, -1.0):
        g = lib.GpuJob(inp)
        g.set_newton_shortcut(shortcut)
        lib._chk(lib.gpu().evpgpu_set_loading(g.ctx, _loading(g, sign)), "set_loading")
        s = _download(g)
        t = 30.0 * np.random.default_rng(3).standard_normal((g.n, 3, 3))
        t = t + t.transpose(0, 2, 1)
        s["sig"] += np.stack([t[:, a, b] for a, b in ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))])
        s["crss"][:] = 4.0
        _upload(g, s)
        _, st = g.run(1, forced=5)
        assert st[0]["ls_trials"] - st[0]["newton_iters"] > 500
        out.append((st[0]["newton_iters"], st[0]["ls_trials"], g.state()))
        g.close()
    assert out[0][:2] == out[1][:2]
    for k in out[0][2]:
        assert np.array_equal(out[0][2][k], out[1][2][k]), k
