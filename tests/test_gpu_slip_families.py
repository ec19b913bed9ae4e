"""The loop's Newton kernel treats the twelve systems of {111}<110> by their
structure and any other set through its Schmid tensors: both against the
oracle's whole loop.  The twelve in another order, with normals and directions
reversed and exchanged ({110}<111> has the same symmetric Schmid tensors), in
each rate law that has such a variant; twelve systems of {112}<111>, and the
twelve with one given twice, which must take the general form.  Bars: those of
the whole-loop parity tests (rounding, carried through three increments)."""
import itertools
import random

import numpy as np
import pytest

import oracle as O
from pyevp import lib, synth
from test_gpu_dd import _compare as _compare_dd
from test_gpu_parity import _compare_jobs

pytestmark = pytest.mark.gpu


def _shuffled():
    rng = random.Random(5)
    out = []
    for n, b in rng.sample(synth.FCC_SLIP, 12):
        if rng.random() < 0.5:
            n = tuple(-c for c in n)
        if rng.random() < 0.5:
            b = tuple(-c for c in b)
        out.append((b, n) if rng.random() < 0.5 else (n, b))
    return out


def _family112():
    out = []
    for b in ((1, 1, 1), (-1, 1, 1), (1, -1, 1), (1, 1, -1)):
        for n in itertools.product((1, -1, 2, -2), repeat=3):
            if sorted(map(abs, n)) == [1, 1, 2] and np.dot(n, b) == 0 and n > (0, 0, 0):
                out.append((n, b))
    assert len(out) == 12
    return out


FAMILIES = {"shuffled": _shuffled(), "112": _family112(), "twice": synth.FCC_SLIP[:11] + synth.FCC_SLIP[:1]}
CASES = [("shuffled", 10.0), ("shuffled", 20.0), ("shuffled", 7.0), ("shuffled", 12.5), ("112", 10.0),
         ("112", 20.0), ("112", 7.0), ("112", 12.5), ("twice", 10.0)]


@pytest.mark.parametrize("family,nrs", CASES)
def test_slip_families_vs_oracle(tmp_path, monkeypatch, family, nrs):
    monkeypatch.setattr(synth, "FCC_SLIP", FAMILIES[family])
    m = synth.Material(nrs=nrs)
    cfg = synth.Config(n=0, dims=(10, 9, 7), grains=5, seed=67, increments=3, pore_fraction=0.02, pore_radius=1,
                       material=m)
    inp = synth.write_job(str(tmp_path), cfg)
    J, g = O.Job(inp), lib.GpuJob(inp)
    _compare_jobs(J, g, 3)
    # the rates of each system, in the file's order and sign
    gd = J.field(O.GAMDOT)
    assert np.abs(g.state()["gamdot"] - gd).max() < 1e-10 * np.abs(gd).max()
    g.close()


def test_slip_families_dislocation_density(tmp_path, monkeypatch):
    monkeypatch.setattr(synth, "FCC_SLIP", FAMILIES["shuffled"])
    cfg = synth.Config(dd=synth.DDLaw(), n=8, grains=8, seed=11, increments=3)
    inp = synth.write_job(str(tmp_path), cfg)
    J, g = O.Job(inp, O.LAW_DD), lib.GpuJob(inp, lib.FP64, law=lib.LAW_DD)
    it_o = J.run(3)
    it_g, _ = g.run(3)
    assert list(it_g) == list(it_o)
    _compare_dd(J, g)
    g.close()
