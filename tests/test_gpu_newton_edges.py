"""Inputs at the edge of what the loop's Newton kernel takes: slip systems
switched off by an infinite CRSS (a file or a caller's state may hold one; the
rate is then 0, the reference's division by infinity), in some voxels of a wave
and in one direction only, or in a whole phase, which is then elastic.  Against
the oracle at the bars of the whole-loop parity tests."""
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
