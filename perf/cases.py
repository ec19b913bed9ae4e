"""Measured cases of the EVPFFT solver: what a user of this package has it do.

Four kinds, each through the package's public entry points:

  loop     one loading increment of a job (GpuJob: input.in, .sx and
           microstructure files) with the fields the writers dump read back;
           IterMax bounds the Green iterations, as it does in the 128^3 run
  newton   the per-voxel stress update on the caller's device buffers
           (evpgpu_newton_device_noalloc)
  adjoint  a calibration step: the macroscopic stress curve of a few
           increments and the gradient of its misfit in the five parameters
  pf       PF_XRX: substeps of the phase-field recrystallisation step

Sizes follow the configurations of pyevp/synth.py (32^3, 64^3 and 128^3 grids
of 64 to 512 grains, 2 % pores, FCC copper, n = 10, uniaxial tension at 1/s),
bench.py (phase field at 128^3, 40 nuclei) and the grids of tests/.

exact() restates the power-law loop and the per-voxel update in 64-bit torch
from their equations (converged Newton solves, torch.fft).
"""
import ctypes as C
import math
import os
import shutil
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "m-themes_amd"))

from pyevp import autograd, lib, pf, synth  # noqa: E402

F64 = torch.float64
DT = 1e-3
TAU0 = 16.0


def listed():
    return [
        # a batch of a few voxels' stress updates: launch and synchronisation latency
        dict(name="newton_1000", kind="newton", n=1000, nrs=10.0),
        # the same on half a 128^3 grid, the higher exponent of the tests
        dict(name="newton_1m", kind="newton", n=1000003, nrs=20.0),
        # the smallest grid the tests run whole: an RVE for a parameter sweep
        dict(name="loop_16_fp64", kind="loop", nx=16, ny=16, nz=16, grains=8, pores=0.0, iters=300,
             precision="fp64", law="power", nrs=10.0, fields="all"),
        # the 32^3 configuration with pores, mixed precision
        dict(name="loop_32_pores_mixed", kind="loop", nx=32, ny=32, nz=32, grains=64, pores=0.02, iters=300,
             precision="mixed", law="power", nrs=10.0, fields="io"),
        # the 64^3 configuration (dense polycrystal), all FP64
        dict(name="loop_64_fp64", kind="loop", nx=64, ny=64, nz=64, grains=128, pores=0.0, iters=200,
             precision="fp64", law="power", nrs=10.0, fields="all"),
        # the 128^3 headline job: 512 grains, 2 % pores, mixed precision
        dict(name="loop_128_pores_mixed", kind="loop", nx=128, ny=128, nz=128, grains=512, pores=0.02, iters=200,
             precision="mixed", law="power", nrs=10.0, fields="io"),
        # a large grid whose planes do not fit one workgroup (the 256^3 run's path)
        dict(name="loop_144x160x160_fp64", kind="loop", nx=144, ny=160, nz=160, grains=512, pores=0.0, iters=50,
             precision="fp64", law="power", nrs=10.0, fields="io"),
        # an image-based RVE: no edge is a power of two, one is odd
        dict(name="loop_45x50x27_mixed", kind="loop", nx=45, ny=50, nz=27, grains=20, pores=0.02, iters=200,
             precision="mixed", law="power", nrs=10.0, fields="io"),
        # the dislocation-density law
        dict(name="loop_64_dd_pores", kind="loop", nx=64, ny=64, nz=64, grains=64, pores=0.02, iters=100,
             precision="fp64", law="dd", nrs=10.0, fields="all"),
        # a calibration step at a non-integral rate exponent
        dict(name="adjoint_24", kind="adjoint", nx=24, ny=24, nz=24, grains=8, increments=2, iters=150, nrs=10.5),
        # recrystallisation of a small, uneven box
        dict(name="pf_48x40x36", kind="pf", nx=48, ny=40, nz=36, grains=24, nuclei=8, steps=8),
        # the 128^3 recrystallisation step of bench.py
        dict(name="pf_128", kind="pf", nx=128, ny=128, nz=128, grains=256, nuclei=40, steps=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


EDGES = (8, 12, 16, 20, 24, 30, 32, 36, 40, 45, 48, 50, 60, 63, 64, 72, 80, 96, 100, 120, 128, 144)


def draw(rng):
    kind = rng.choice(["loop", "loop", "loop", "loop", "newton", "newton", "adjoint", "pf", "pf"])
    if kind == "newton":
        return dict(kind=kind, n=_log_int(rng, 64, 1500000), nrs=rng.choice([5.0, 10.0, 10.0, 12.5, 20.0]))
    if kind == "adjoint":
        e = rng.choice([8, 12, 16, 24, 32])
        return dict(kind=kind, nx=e, ny=e, nz=e, grains=rng.randint(4, 16), increments=rng.choice([1, 2, 3]),
                    iters=rng.randint(50, 150), nrs=rng.choice([10.0, 10.5, 8.25]))
    if kind == "pf":
        nx, ny, nz = (_log_int(rng, 8, 128) for _ in range(3))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, grains=max(3, nx * ny * nz // 8192), nuclei=rng.randint(2, 40),
                    steps=rng.randint(2, 10))
    if rng.random() < 0.6:  # a cube, as most runs are
        nx = ny = nz = rng.choice([16, 24, 32, 48, 64, 80, 96, 120, 128])
    else:
        nx, ny, nz = (rng.choice(EDGES) for _ in range(3))
    n = nx * ny * nz
    law = rng.choice(["power", "power", "power", "dd"])
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, grains=max(4, n // 4096), pores=rng.choice([0.0, 0.02, 0.04]),
                iters=max(20, min(rng.randint(60, 250), int(2.5e8 / n))),
                precision="fp64" if law == "dd" else rng.choice(["fp64", "mixed"]), law=law,
                nrs=rng.choice([10.0, 10.0, 10.0, 20.0, 12.5]), fields=rng.choice(["io", "io", "all"]) if n < 3e5 else "io")


# ---------------------------------------------------------------- inputs --
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _euler(rng, m):
    """m uniform SO(3) orientations as Bunge angles in degrees, as the files hold them"""
    u = rng.uniform(0.0, 1.0, (m, 3))
    return np.round(np.stack([360.0 * u[:, 0], np.degrees(np.arccos(2.0 * u[:, 1] - 1.0)), 360.0 * u[:, 2]], 1), 8)


def _voronoi(shape, seeds):
    """periodic Voronoi labels (0-based) of the voxel points"""
    d = _dev()
    ax = [torch.arange(n, dtype=F64, device=d) for n in shape]
    best = torch.full(shape, math.inf, dtype=F64, device=d)
    lab = torch.zeros(shape, dtype=torch.int32, device=d)
    for g, s in enumerate(seeds):
        q = []
        for m in range(3):
            a = (ax[m] - float(s[m])).abs()
            q.append(torch.minimum(a, shape[m] - a) ** 2)
        r = q[0][:, None, None] + q[1][None, :, None] + q[2][None, None, :]
        new = r < best
        best = torch.where(new, r, best)
        lab = torch.where(new, torch.full_like(lab, g), lab)
    return lab


def _spheres(shape, centres, r2):
    d = _dev()
    ax = [torch.arange(n, dtype=torch.int64, device=d) for n in shape]
    for c in centres:
        q = []
        for m in range(3):
            a = (ax[m] - int(c[m])).abs()
            q.append(torch.minimum(a, shape[m] - a) ** 2)
        yield (q[0][:, None, None] + q[1][None, :, None] + q[2][None, None, :]) <= r2


def _structure(case, seed):
    """(Euler angles of the grains, label[N], gas[N]) of a case's polycrystal"""
    rng = np.random.default_rng([seed, 1])
    shape = (case["nx"], case["ny"], case["nz"])
    eul = _euler(rng, case["grains"])
    lab = _voronoi(shape, rng.uniform(0.0, 1.0, (case["grains"], 3)) * np.array(shape))
    gas = torch.zeros(shape, dtype=torch.bool, device=lab.device)
    frac = case.get("pores", 0.0)
    if frac > 0.0:  # spheres of radius 3 (123 voxels), radius 2 (33) on thin grids
        r2, vol = (9, 123) if min(shape) >= 12 else (4, 33)
        m = max(1, int(round(frac * math.prod(shape) / vol)))
        for s in _spheres(shape, rng.integers(0, np.array(shape), (m, 3)), r2):
            gas |= s
    return eul, lab.reshape(-1).cpu().numpy(), gas.reshape(-1).cpu().numpy()


def _write_ms(path, shape, eul, grain, phase):
    """synth.write_ms's file with its columns padded to fixed widths; eul[g - 1]
    are grain g's angles"""
    def column(texts, w):
        return np.frombuffer("".join(t.rjust(w) for t in texts).encode(), dtype=np.uint8).reshape(-1, w)

    m = int(grain.max())
    angles = column(["%.8f %.8f %.8f" % (tuple(eul[g]) if g < len(eul) else (0.0, 0.0, 0.0)) for g in range(m)], 40)
    ax = [column([str(i + 1) for i in range(n)], 4) for n in shape]
    out = np.empty(tuple(shape) + (62,), dtype=np.uint8)
    out[..., 0:40] = angles[grain.reshape(shape) - 1]
    out[..., 40:44] = ax[0][:, None, None]
    out[..., 44:48] = ax[1][None, :, None]
    out[..., 48:52] = ax[2][None, None, :]
    out[..., 52:59] = column([str(g + 1) for g in range(m)], 7)[grain.reshape(shape) - 1]
    out[..., 59:61] = column(["1", "2"], 2)[phase.reshape(shape) - 1]
    out[..., 61] = ord("\n")
    out.tofile(path)


def _material(case):
    return synth.Material(nrs=float(case["nrs"]))


def _open(case, seed):
    """the case's job, from files in the reference's formats"""
    shape = (case["nx"], case["ny"], case["nz"])
    eul, lab, gas = _structure(case, seed)
    cfg = synth.Config(n=shape[0], dims=shape, grains=case["grains"], increments=100, dt=DT, err=1e-8,
                       iter_max=case["iters"], pore_fraction=case.get("pores", 0.0), material=_material(case),
                       dd=synth.DDLaw() if case.get("law") == "dd" else None)
    grain, phase = (lab + 1).astype(np.int32), np.ones(lab.size, np.int32)
    grain[gas], phase[gas] = case["grains"] + 1, 2
    d = tempfile.mkdtemp(prefix="evpcase_")
    try:
        _write_ms(os.path.join(d, "ms.txt"), shape, eul, grain, phase)
        synth.write_sx(os.path.join(d, "Cu.sx"), cfg.material)
        inp = os.path.join(d, "input.in")
        synth.write_input(inp, cfg)
        return lib.GpuJob(inp, lib.MIXED if case.get("precision") == "mixed" else lib.FP64,
                          law=lib.LAW_DD if case.get("law") == "dd" else lib.LAW_POWER)
    finally:
        shutil.rmtree(d, ignore_errors=True)


FIELDS = (("sig", 6), ("disgrad", 9), ("eps", 6), ("edot", 6), ("tran", 9), ("crss", 24), ("gamacum", 1),
          ("gamdot", 12))
IO_FIELDS = ("sig", "eps", "edot")  # what the .iout writers dump


def _newton_inputs(case, seed):
    """Voxel states near yield in a polycrystal of 64 orientations.  The
    strain is chosen so that the stress sigma* solves the update from lambda
    (a disturbance of sigma* between 1e-3 and 3 MPa)."""
    g = torch.Generator(device=_dev()).manual_seed(int(seed))
    rng = np.random.default_rng([seed, 2])
    n, d = case["n"], _dev()
    P = _Power(_material(case))
    eul = _euler(rng, 64)
    cgr = P.c_grains(eul)
    c0 = cgr.mean(0)
    sgr, s0 = np.linalg.inv(cgr), np.linalg.inv(c0)
    o = torch.randint(0, 64, (n,), generator=g, device=d)
    rand = lambda *s: torch.randn(*s, generator=g, device=d, dtype=F64)  # noqa: E731
    R = torch.as_tensor(_rot(eul), device=d)[o]  # crystal -> sample, as update_orient leaves it
    spin = 1e-2 * rand(n, 3)
    W = torch.zeros(n, 3, 3, device=d, dtype=F64)
    W[:, 0, 1], W[:, 0, 2], W[:, 1, 2] = spin[:, 0], spin[:, 1], spin[:, 2]
    R = torch.linalg.matrix_exp(W - W.transpose(1, 2)) @ R
    crss = TAU0 + 6.0 * torch.rand(24, n, generator=g, device=d, dtype=F64)
    star = 18.0 * rand(6, n)  # B-basis: about 45 MPa von Mises
    star[5] += 20.0
    lam = star + 10.0 ** (-3.0 + 3.5 * torch.rand(1, n, generator=g, device=d, dtype=F64)) * rand(6, n)
    eps = torch.zeros(6, n, device=d, dtype=F64)
    eps[:5] = 1e-3 * rand(5, n)
    m = P.schmid(R)
    ed, gd, _ = P.rate(m, star, crss.reshape(12, 2, n))
    t = torch.as_tensor(s0, device=d) @ (lam - star)
    E = eps + DT * ed + torch.einsum("nij,jn->in", torch.as_tensor(sgr, device=d)[o], star) - t
    return dict(eul=eul, o=o, sgr=sgr, R=R, crss=crss, star=star, lam=lam, eps=eps, E=E, ed=ed, gd=gd, t=t)


class _State:
    """what a case's program holds; its device handles go with it"""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for h in ("job", "pf"):
            if getattr(self, h, None) is not None:
                getattr(self, h).close()


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pf":
        shape = (case["nx"], case["ny"], case["nz"])
        rng = np.random.default_rng([seed, 3])
        gid = _voronoi(shape, rng.uniform(0.0, 1.0, (case["grains"], 3)) * np.array(shape)) + 1
        rho = torch.as_tensor(200.0 + rng.uniform(0.0, 50.0, shape), device=gid.device)
        for k, s in enumerate(_spheres(shape, rng.integers(0, np.array(shape), (case["nuclei"], 3)), 5)):
            gid[s] = case["grains"] + 1 + k
            rho[s] = 96.0
        return _State(kind=kind, pf=pf.PhaseField(shape, 60000), gid=gid.to(torch.int32).cpu().numpy(),
                      rho=rho.cpu().numpy(), steps=case["steps"], params=synth.pf_params(case["grains"]),
                      rho_avg=np.zeros(60000))
    if kind == "newton":
        n = case["n"]
        q = _newton_inputs(case, seed)
        # a job whose grains are the batch's orientations gives the context its
        # material and loading: <C> is the mean over them
        job = _open_cells(case, q["eul"])
        f = lib.gpu().evpgpu_newton_device_noalloc
        f.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int] + [C.c_void_p] * 9
        f.restype = C.c_int
        d = q["lam"].device
        s = _State(kind=kind, job=job, f=f, n=n, phase=torch.ones(n, dtype=torch.int32, device=d),
                   orient=q["o"].to(torch.int32), sgr=torch.as_tensor(q["sgr"].reshape(-1), device=d),
                   lam=_sym(q["lam"]), E=_sym(q["E"]), eps=_sym(q["eps"]),
                   tran=q["R"].reshape(n, 9).t().contiguous(), crss=q["crss"].contiguous(),
                   sig=torch.empty(6, n, dtype=F64, device=d), edot=torch.zeros(6, n, dtype=F64, device=d),
                   gamdot=torch.zeros(12, n, dtype=F64, device=d), err=torch.zeros(n, 2, dtype=F64, device=d),
                   niter=torch.zeros(n, dtype=torch.int32, device=d))
        if d.type == "cuda":
            torch.cuda.synchronize()
        return s
    job = _open(case, seed)
    if kind == "adjoint":
        p = torch.tensor([TAU0, 10.0, 200.0, 20.0, float(case["nrs"])], dtype=F64)
        return _State(kind=kind, job=job, params=p, n=case["increments"],
                      target=torch.as_tensor(np.random.default_rng([seed, 4]).uniform(20.0, 60.0, case["increments"])))
    names = IO_FIELDS if case["fields"] == "io" else [f for f, _ in FIELDS]
    pin = torch.cuda.is_available()
    bufs = {f: torch.zeros(m * job.n, dtype=F64, pin_memory=pin).numpy() for f, m in FIELDS if f in names}
    return _State(kind=kind, job=job, bufs=bufs)


def _open_cells(case, eul):
    """8 x 8 x 8 voxels, every 8 of them one of the 64 orientations"""
    d = tempfile.mkdtemp(prefix="evpcase_")
    try:
        lab = np.repeat(np.arange(64), 8)
        cfg = synth.Config(n=8, grains=64, increments=1, dt=DT, material=_material(case))
        synth.write_ms(os.path.join(d, "ms.txt"), 8, eul[lab], (lab + 1).astype(np.int32), np.ones(512, np.int32))
        synth.write_sx(os.path.join(d, "Cu.sx"), cfg.material)
        synth.write_input(os.path.join(d, "input.in"), cfg)
        return lib.GpuJob(os.path.join(d, "input.in"), lib.FP64)
    finally:
        shutil.rmtree(d, ignore_errors=True)


# ------------------------------------------------------------------- run --
def run(s):
    if s.kind == "pf":
        gid, rho_avg = s.pf.pf_xrx(s.gid, s.rho, s.steps, s.params, s.rho_avg)
        return dict(gid=gid, rho_avg=rho_avg)
    if s.kind == "newton":
        s.sig.copy_(s.lam)
        torch.cuda.current_stream().synchronize()  # the update runs on the context's own stream
        st = s.f(s.job.ctx, s.n, _ptr(s.phase), _ptr(s.orient), _ptr(s.sgr), 64, _ptr(s.sig), _ptr(s.E), _ptr(s.eps),
                 _ptr(s.tran), _ptr(s.crss), _ptr(s.edot), _ptr(s.gamdot), _ptr(s.err), _ptr(s.niter))
        if st:
            raise lib.EvpError(st, "evpgpu_newton_device_noalloc")
        return dict(sig=s.sig, edot=s.edot, gamdot=s.gamdot, err=s.err, niter=s.niter)
    if s.kind == "adjoint":
        p = s.params.clone().requires_grad_(True)
        curve = autograd.MacroStressCurve.apply(p, s.job, s.n, 0, 5, 1e-12, 4000)
        ((curve[:, 2] - s.target) ** 2).sum().backward()
        return dict(curve=curve.detach(), grad=p.grad)
    iters, _ = s.job.run(1)
    lib._chk(lib.gpu().evpgpu_download_state(s.job.ctx, *[lib._p(s.bufs[f]) if f in s.bufs else None
                                                          for f, _ in FIELDS]), "download_state")
    m = s.job.macro()
    return dict(s.bufs, iters=iters, **{k: m[k] for k in ("sig_avg", "eps_avg", "edot_avg", "disgrad_avg_t")})


# ------------------------------------------------------------------ work --
def work(case):
    """Bytes and operations of one pass.  Loop, per voxel and Green iteration:
    the update reads sigma, E, eps, the rotation, 12 CRSS and the two indices
    and writes sigma; E is updated in place; the half spectrum goes out and
    back once (x lines cross the planes).  Operations: 5.1 kflop of the update
    (two Newton iterations), 12 real transforms of 2.5 log2(N), 0.2 kflop of
    the Green operator.  Phase field: per voxel and substep a list of about
    1.6 entries (12 B each), its grain and its stored energy, read and written."""
    kind = case["kind"]
    if kind == "newton":
        return dict(bytes=case["n"] * 8.0 * (6 + 6 + 6 + 9 + 24 + 1 + 6 + 6 + 12 + 2.5), flops=case["n"] * 7.5e3)
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "pf":
        return dict(bytes=2.0 * n * case["steps"] * (1.6 * 12 + 4 + 4 + 8), flops=1e2 * n * case["steps"])
    it = case["iters"] * (case["increments"] if kind == "adjoint" else 1)
    spec = 2 * 24.5 if case.get("precision") == "mixed" else 2 * 49.0
    solid = 1.0 - case.get("pores", 0.0)
    b = (solid * (4 * 48 + 72 + 96 + 8) + 2 * 48 + spec) * n * it
    f = (solid * 5.1e3 + 12 * 2.5 * math.log2(n) + 200.0) * n * it
    return dict(bytes=b, flops=f)


# ----------------------------------------------------------------- exact --
r2, r3, r6 = 1 / math.sqrt(2), 1 / math.sqrt(3), 1 / math.sqrt(6)
BASIS = np.zeros((6, 3, 3))
BASIS[0] = np.diag([-r2, r2, 0])
BASIS[1] = np.diag([-r6, -r6, 2 * r6])
for _i, (_a, _b) in enumerate(((1, 2), (0, 2), (0, 1))):
    BASIS[2 + _i, _a, _b] = BASIS[2 + _i, _b, _a] = r2
BASIS[5] = r3 * np.eye(3)
IJ = ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))
PI = 3.14159265359  # the reference's value: degrees to radians


def _rot(eul):
    """rotations crystal -> sample [m, 3, 3] of Bunge angles in degrees"""
    p1, P, p2 = (np.asarray(eul, dtype=np.float64) * (PI / 180.0)).T
    c1, s1, c, s, c2, s2 = np.cos(p1), np.sin(p1), np.cos(P), np.sin(P), np.cos(p2), np.sin(p2)
    g = np.array([[c1 * c2 - s1 * s2 * c, s1 * c2 + c1 * s2 * c, s2 * s],
                  [-c1 * s2 - s1 * c2 * c, -s1 * s2 + c1 * c2 * c, c2 * s],
                  [s1 * s, -c1 * s, c]])
    return np.ascontiguousarray(g.transpose(2, 1, 0))


def _sym(v):
    """B-basis [6, n] -> symmetric components 11 22 33 23 13 12"""
    T = torch.as_tensor(np.array([[BASIS[i, a, b] for i in range(6)] for a, b in IJ]), device=v.device)
    return (T @ v).contiguous()


def _vec(t):
    """symmetric components -> B-basis"""
    T = torch.as_tensor(np.array([[BASIS[i, a, b] * (1 if a == b else 2) for a, b in IJ] for i in range(6)]),
                        device=t.device)
    return T @ t


class _Power:
    """FCC power-law crystal in 64-bit torch: voxels along the last axis"""

    def __init__(self, m):
        self.n, self.g0 = m.nrs, m.gam0
        c = np.zeros((3, 3, 3, 3))
        for i in range(3):
            c[i, i, i, i] = m.c11
            for j in range(3):
                if i != j:
                    c[i, i, j, j] = m.c12
                    c[i, j, i, j] = c[i, j, j, i] = m.c44
        self.c = c
        nb = np.array(synth.FCC_SLIP, dtype=np.float64)
        self.nv, self.bv = nb[:, 0] / math.sqrt(3.0), nb[:, 1] / math.sqrt(2.0)

    def c_grains(self, eul):
        """stiffness [m, 6, 6] of each orientation in the B-basis"""
        out = []
        for R in _rot(eul):
            c = np.einsum("im,jn,kp,lq,mnpq->ijkl", R, R, R, R, self.c, optimize=True)
            out.append(np.einsum("iab,abcd,jcd->ij", BASIS, c, BASIS, optimize=True))
        return np.array(out)

    def schmid(self, R):
        """Schmid tensors [12, 5, n] of rotations [n, 3, 3]"""
        B = torch.as_tensor(BASIS[:5], device=R.device)
        out = torch.empty(12, 5, R.shape[0], dtype=F64, device=R.device)
        for s in range(12):
            tn = R @ torch.as_tensor(self.nv[s], device=R.device)
            tb = R @ torch.as_tensor(self.bv[s], device=R.device)
            p = 0.5 * (tn[:, :, None] * tb[:, None, :] + tb[:, :, None] * tn[:, None, :])
            out[s] = torch.einsum("iab,nab->in", B, p)
        return out

    def rate(self, m, s, crss):
        """(edot [6, n], shear rates [12, n], their derivatives) at stress s;
        crss [12, n] or, by direction, [12, 2, n]"""
        tau = (m * s[None, :5]).sum(1)
        cr = crss if crss.dim() == 2 else torch.where(tau < 0, crss[:, 1], crss[:, 0])
        x = tau / cr
        p = self.g0 * x.abs() ** (self.n - 1.0)
        gd = p * x
        ed = torch.zeros_like(s)
        ed[:5] = (m * gd[:, None]).sum(0)
        return ed, gd, self.n * p / cr

    def update(self, m, lam, bp, crss, S, C0, S0):
        """the stress solving s - lam + C0 (bp + dt edot(s) + S s) = 0;
        S a list of 21 per-voxel entries (upper triangle, row by row)"""
        tri = [(i, j) for i in range(6) for j in range(i, 6)]
        full = {}
        for (i, j), v in zip(tri, S):
            full[i, j] = full[j, i] = v

        def mismatch(s):
            ed, gd, dg = self.rate(m, s, crss)
            t = bp + DT * ed
            for i in range(6):
                for j in range(6):
                    t[i] += full[i, j] * s[j]
            return t, dg

        s = lam.clone()
        t, dg = mismatch(s)
        res = s - lam + C0 @ t
        f = (res * res).sum(0)
        for _ in range(60):
            b = S0 @ res
            w = DT * dg
            k = {}
            for i, j in tri:
                k[i, j] = full[i, j] + S0[i, j]
                if j < 5:
                    k[i, j] = k[i, j] + (m[:, i] * m[:, j] * w).sum(0)
            # Cholesky K = L L^T, then the step
            L, inv = {}, []
            for j in range(6):
                d = k[j, j] - sum(L[j, q] ** 2 for q in range(j))
                inv.append(d.rsqrt())
                for i in range(j + 1, 6):
                    L[i, j] = (k[j, i] - sum(L[i, q] * L[j, q] for q in range(j))) * inv[j]
            y = []
            for i in range(6):
                y.append((b[i] - sum(L[i, q] * y[q] for q in range(i))) * inv[i])
            x = [None] * 6
            for i in range(5, -1, -1):
                x[i] = (y[i] - sum(L[q, i] * x[q] for q in range(i + 1, 6))) * inv[i]
            step = -torch.stack(x)
            step *= torch.clamp(10.0 / step.norm(dim=0).clamp(min=1e-300), max=1.0)
            small = step.abs().max(0).values / s.abs().max(0).values.clamp(min=1.0)
            a = torch.ones_like(f)
            for _ in range(30):  # backtracking, off once the merit is down to rounding
                s1 = s + a * step
                t, dg = mismatch(s1)
                res1 = s1 - lam + C0 @ t
                f1 = (res1 * res1).sum(0)
                worse = (f1 > f) & (small > 1e-9)
                if not bool(worse.any()):
                    break
                a = torch.where(worse, 0.5 * a, a)
            s, res, f = s1, res1, f1
            if float(small.max()) < 1e-13 or not s.numel():
                break
        return s


def _directions(shape, device):
    """unit wave vectors [3, nx, ny, nz/2+1] of the half spectrum and of -k"""
    def xi(neg):
        out = []
        for m, n in enumerate(shape):
            k = np.arange(n // 2 + 1 if m == 2 else n)
            if neg:
                k = (n - k) % n
            x = k * (1.0 / n)
            x = x - np.where(2 * k == n, 1.0, np.round(x))  # Nyquist to -1/2
            out.append(torch.as_tensor(x, dtype=F64, device=device))
        g = torch.stack(torch.meshgrid(*out, indexing="ij"))
        return g / g.norm(dim=0).clamp(min=1e-300)
    return xi(False), xi(True)


def _exact_loop(case, seed):
    d = _dev()
    shape = (case["nx"], case["ny"], case["nz"])
    N = math.prod(shape)
    eul, lab, gas = _structure(case, seed)
    P = _Power(_material(case))
    cgr = P.c_grains(eul)
    solid = np.where(~gas)[0]
    cnt = np.bincount(lab[solid], minlength=len(eul))
    c0n = np.einsum("g,gij->ij", cnt / N, cgr)
    s0n = np.linalg.inv(c0n)
    C0, S0 = torch.as_tensor(c0n, device=d), torch.as_tensor(s0n, device=d)
    c4 = np.einsum("ij,iab,jcd->abcd", c0n, BASIS, BASIS, optimize=True)
    s4 = np.einsum("ij,iab,jcd->abcd", s0n, BASIS, BASIS, optimize=True)
    vel, flag, stress = np.zeros((3, 3)), (0, 0, 1, 1, 1, 1), (1, 1, 0, 0, 0, 0)
    vel[2, 2] = 1.0
    idx = torch.as_tensor(solid, device=d)
    og = torch.as_tensor(lab[solid].astype(np.int64), device=d)
    nv = idx.numel()
    m = P.schmid(torch.as_tensor(_rot(eul), device=d))[:, :, og]
    Sg = torch.as_tensor(np.linalg.inv(cgr), device=d)
    S = [Sg[:, i, j][og] for i in range(6) for j in range(i, 6)]
    e0 = np.array([vel[a, b] * DT for a, b in IJ])
    v0 = np.einsum("iab,ab->i", BASIS, vel * DT)
    sig = torch.zeros(6, N, dtype=F64, device=d)
    sig[:, idx] = _sym(torch.as_tensor(np.einsum("gij,j->ig", cgr, v0), device=d)[:, og].contiguous())
    E = torch.as_tensor(e0, device=d)[:, None].expand(6, N).clone()
    crss = torch.full((12, nv), TAU0, dtype=F64, device=d)
    dirs = _directions(shape, d)
    T = torch.as_tensor(c4, device=d)
    om = []
    for n in dirs:
        A = torch.einsum("ijkl,jxyz,lxyz->xyzik", T, n, n)
        A[0, 0, 0] = torch.eye(3, dtype=F64, device=d)
        om.append(torch.linalg.inv(A).permute(3, 4, 0, 1, 2).contiguous())
        del A
    dD, acum = np.zeros((3, 3)), np.zeros((3, 3))
    for _ in range(case["iters"]):
        h = torch.fft.rfftn(sig.reshape(6, *shape), dim=(1, 2, 3))
        e = torch.zeros_like(h)
        full = {}
        for c, (a, b) in enumerate(IJ):
            full[a, b] = full[b, a] = h[c]
        for n, O in zip(dirs, om):
            t = [sum(full[k, l] * n[l] for l in range(3)) for k in range(3)]
            u = [sum(O[i, k] * t[k] for k in range(3)) for i in range(3)]
            for c, (a, b) in enumerate(IJ):
                e[c] -= 0.25 * (u[a] * n[b] + u[b] * n[a])
        e[:, 0, 0, 0] = 0
        del h, full, t, u
        # k = 0 holds no strain: the mean follows the boundary conditions
        E += torch.fft.irfftn(e, s=shape, dim=(1, 2, 3)).reshape(6, N)
        E += torch.as_tensor(np.array([0.5 * (dD[a, b] + dD[b, a]) for a, b in IJ]), device=d)[:, None]
        del e
        lam = _vec(sig[:, idx])
        s = P.update(m, lam, -_vec(E[:, idx]), crss, S, C0, S0)
        sig[:, idx] = _sym(s)
        avg = sig.mean(1).cpu().numpy()
        dD = np.zeros((3, 3))
        for i, (a, b) in enumerate(IJ):
            if flag[i] == 0:
                dD[a, b] = sum(s4[a, b, k, l] * stress[q] * (0.0 - avg[q]) for q, (k, l) in enumerate(IJ))
        acum += dD
    ed = torch.zeros(6, N, dtype=F64, device=d)
    ed[:, idx] = _sym(P.rate(m, s, crss)[0])

    def tensor(v):
        t = np.zeros((3, 3))
        for c, (a, b) in enumerate(IJ):
            t[a, b] = t[b, a] = float(v[c])
        return t

    flat = lambda x: x.reshape(-1).cpu().numpy()  # noqa: E731
    out = dict(sig=flat(sig), eps=flat(ed * DT), edot=flat(ed), iters=None, sig_avg=tensor(sig.mean(1)),
               eps_avg=tensor(ed.mean(1) * DT), edot_avg=tensor(ed.mean(1)), disgrad_avg_t=vel * DT + acum)
    if case["fields"] == "all":
        out.update({f: None for f, _ in FIELDS if f not in IO_FIELDS})
    return out


def exact(case, seed):
    if case["kind"] == "newton":
        q = _newton_inputs(case, seed)
        s0 = q["star"] - q["lam"]
        return dict(sig=_sym(q["star"]), edot=_sym(q["ed"]), gamdot=q["gd"],
                    err=torch.stack([s0.norm(dim=0), q["t"].norm(dim=0)], 1), niter=None)
    # the loop's power law; a longer loop on a large grid takes over 20 seconds here
    if case["kind"] == "loop" and case["law"] == "power" and case["iters"] * case["nx"] * case["ny"] * case["nz"] < 4.5e8:
        return _exact_loop(case, seed)
    return None
