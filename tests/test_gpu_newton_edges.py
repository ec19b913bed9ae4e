"""Inputs at the edge of what the loop's Newton kernel takes: slip systems
switched off by an infinite CRSS (a file or a caller's state may hold one; the
rate is then 0, the reference's division by infinity), in some voxels of a wave
and in one direction only, or in a whole phase, which is then elastic, against
the oracle at the bars of the whole-loop parity tests; a C0 that is not
positive definite, as a caller may set one; and rate laws so steep that the
tangent's terms span more than the 16 digits of its sums."""
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


@pytest.mark.parametrize("nrs", [50.0, 50.5])
def test_steep_rates_next_to_pores(job_factory, nrs):
    """The first iteration's overstress next to pores at a steep rate law: its
    tangent's weights span more than 1e16, and rounded sums of them need not be
    positive definite.  The same stresses as the batch update's, from the same
    inputs, to where both end (steps below 1e-7 of the stress: a bar of 1e-6);
    then more iterations of the loop."""
    inp = job_factory(f"steep{nrs}", n=16, grains=8, seed=25, increments=1, pore_fraction=0.04, pore_radius=2,
                      material=synth.Material(nrs=nrs))
    J, g = O.Job(inp), lib.GpuJob(inp)
    solid = np.where(J.phase() == 1)[0]
    m = solid.size
    a = {k: np.ascontiguousarray(v[:, solid]) for k, v in _download(g).items()}
    g.run(1, forced=1)
    b = {k: v[:, solid] for k, v in _download(g).items()}
    d = b["disgrad"]
    E = np.stack([d[0], d[4], d[8], (d[5] + d[7]) / 2, (d[2] + d[6]) / 2, (d[1] + d[3]) / 2])
    ctx = lib.Context.__new__(lib.Context)
    ctx.h = g.ctx
    st, sig, *_ = ctx.newton(np.ones(m, np.int32), np.arange(m, dtype=np.int32), np.linalg.inv(J.cgr()[solid]), a["sig"], E,
                             a["eps"], a["tran"], a["crss"])
    ctx.h = None
    assert st == 0
    assert np.abs(b["sig"] - sig).max() < 1e-6 * np.abs(sig).max()
    g.reset()
    g.run(1, forced=30)
    assert np.isfinite(g.state()["Sig"]).all()
    g.close()
