"""Performance cases of the library: what its callers have it compute.

Each case is one call (or one time step's call) through a public entry point:

  p3d        cvtx_hip_p3d_eval: 3D particles resident on the GPU (velocity,
             stretching, viscous exchange, any subset in one pass)
  p2d        cvtx_hip_p2d_eval: 2D particles resident on the GPU
  f3d        cvtx_hip_f3d_eval: straight filaments on particles
  clouds     cvtx_hip_batch_eval: many independent 3D clouds, one launch
  relax      cvtx_hip_relax_eval: Pedrizzetti relaxation, strengths in place
  vort       cvtx_hip_vort_eval: vorticity field at points
  influence  cvtx_hip_f3d_inf_eval: filament influence matrix
  host       the reference API on host arrays (cvtx_P3D_M2M_vel and others)
  remesh     cvtx_P3D_redistribute_on_grid / cvtx_P2D_... on host arrays

The fields are the ones of cvortex_amd/workloads.py (uniform cube, thin vortex
ring, horseshoe lattice, uneven clouds, 2D sheet) and of the reference's
agreement tests (a box of uniformly random particles), drawn here from a seed
so that any size can be made quickly.
"""
import ctypes
import math

import numpy as np
import torch

import cvortex_amd as cv
from cvortex_amd import device as D
from cvortex_amd.types import (P2D_DTYPE, P3D_DTYPE, REG_ID, make_f3d, make_p2d, make_p3d,
                               pointer_array)

RING_R, RING_CORE, RING_SIGMA = 1.0, 0.05, 0.02
FDT = 0.1            # relaxation factor
NU = 1e-3            # kinematic viscosity
REGS = ("singular", "winckelmans", "planetary", "gaussian")


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------

def listed():
    return [
        # the smallest calls: a program of the reference API with a thousand
        # particles (the size of the reference's own agreement tests), host
        # arrays in and out, one call per step
        dict(name="host_vel_1000", kind="host", fn="P3D_vel", n_src=1000, n_tgt=1000,
             reg="winckelmans"),
        # a small cloud resident on the GPU: velocity of every particle
        dict(name="cube_8192_vel", kind="p3d", field="cube", n_src=8192, n_tgt=0,
             reg="winckelmans", vel=True, dvort=False, visc=False, acc=1),
        # all three right-hand sides of a viscous step, sources and targets of
        # different, odd counts
        dict(name="box_ragged_visc", kind="p3d", field="box", n_src=23011, n_tgt=9973,
             reg="winckelmans", vel=True, dvort=True, visc=True, acc=1),
        # a vortex ring of ordinary size, one inviscid step's right-hand side
        dict(name="ring_65536", kind="p3d", field="ring", n_src=65536, n_tgt=0, reg="gaussian",
             vel=True, dvort=True, visc=False, acc=1),
        # the headline workload, the largest
        dict(name="ring_1048576", kind="p3d", field="ring", n_src=1 << 20, n_tgt=0, reg="gaussian",
             vel=True, dvort=True, visc=False, acc=1),
        # many uneven clouds in one persistent launch (an ensemble)
        dict(name="clouds_128", kind="clouds", n_clouds=128, lo=1024, hi=65536,
             reg="winckelmans", acc=2),
        # a vortex lattice acting on a particle wake
        dict(name="lattice_wake", kind="f3d", nx=128, ny=128, n_tgt=1 << 20, vel=True,
             dvort=True),
        # a 2D sheet: point-vortex velocity of an inviscid step
        dict(name="sheet_262144", kind="p2d", n=262144, reg="planetary", visc=False),
        # the same sheet's viscous step, an odd count
        dict(name="sheet_visc_100003", kind="p2d", n=100003, reg="gaussian", visc=True),
        # divergence control of a ring between steps
        dict(name="relax_1048576", kind="relax", n=1 << 20, reg="gaussian"),
        # the matrix of a 128 x 128 panel vortex lattice
        dict(name="influence_16384", kind="influence", nx=128, ny=128, n_mes=16384),
        # remeshing of the ring, host arrays in and out
        dict(name="remesh_1048576", kind="remesh", dim=3, n=1 << 20, fn="m4p", h=0.01),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("p3d", "p3d", "p2d", "f3d", "clouds", "relax", "vort", "influence", "host",
                       "remesh"))
    if kind == "p3d":
        reg = rng.choice(REGS)
        visc = reg in ("winckelmans", "gaussian") and rng.random() < 0.4
        vel = rng.random() < 0.75
        dvort = visc or not vel or rng.random() < 0.5
        return dict(kind=kind, field=rng.choice(("cube", "ring", "box")),
                    n_src=_logint(rng, 300, 500000),
                    n_tgt=0 if rng.random() < 0.5 else _logint(rng, 300, 500000), reg=reg,
                    vel=vel or (visc and not dvort), dvort=dvort, visc=visc,
                    acc=rng.choice((1, 1, 1, 2)))
    if kind == "p2d":
        reg = rng.choice(REGS)
        return dict(kind=kind, n=_logint(rng, 500, 600000), reg=reg,
                    visc=reg in ("winckelmans", "gaussian") and rng.random() < 0.6)
    if kind == "f3d":
        vel = rng.random() < 0.7
        return dict(kind=kind, nx=_logint(rng, 16, 160), ny=_logint(rng, 16, 160),
                    n_tgt=_logint(rng, 1000, 1000000), vel=vel,
                    dvort=not vel or rng.random() < 0.6)
    if kind == "clouds":
        return dict(kind=kind, n_clouds=_logint(rng, 8, 160), lo=_logint(rng, 200, 2000),
                    hi=_logint(rng, 4000, 50000), reg=rng.choice(("winckelmans", "gaussian")),
                    acc=rng.choice((1, 2)))
    if kind == "relax":
        return dict(kind=kind, n=_logint(rng, 2000, 1000000), reg=rng.choice(("winckelmans", "gaussian")))
    if kind == "vort":
        return dict(kind=kind, n_src=_logint(rng, 2000, 600000), n_tgt=_logint(rng, 1000, 600000),
                    reg=rng.choice(("winckelmans", "gaussian")))
    if kind == "influence":
        nx, ny = _logint(rng, 12, 150), _logint(rng, 12, 150)
        return dict(kind=kind, nx=nx, ny=ny, n_mes=_logint(rng, 200, 20000))
    if kind == "host":
        fn = rng.choice(("P3D_vel", "P3D_vel", "P3D_dvort", "P3D_visc", "P2D_vel", "F3D_vel",
                         "P3D_vort"))
        reg = rng.choice(("winckelmans", "gaussian")) if fn in ("P3D_visc", "P3D_vort") else rng.choice(REGS)
        return dict(kind=kind, fn=fn, n_src=_logint(rng, 600, 30000), n_tgt=_logint(rng, 600, 30000),
                    reg=reg)
    dim = rng.choice((3, 3, 2))
    return dict(kind="remesh", dim=dim, n=_logint(rng, 5000, 1000000),
                fn=rng.choice(("m4p", "m4p", "lambda1", "lambda2", "lambda3")),
                h=round(rng.uniform(0.008, 0.03), 4))


# --------------------------------------------------------------------------
# fields
# --------------------------------------------------------------------------

class _Gpu:
    """A torch tensor as the device-resident wrappers take it."""

    def __init__(self, t):
        self.t = t

    @property
    def addr(self):
        return self.t.data_ptr()


def _gen(seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(0x5EED0000 + int(seed))
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=g.device, dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=g.device, dtype=torch.float64)


def _points3(field, n, g):
    """(coordinates (n, 3), strengths (n, 3), volumes (n)) in FP64."""
    if field == "cube":          # uniform in [-1, 1]^3, random strengths
        return 2.0 * _rand(g, n, 3) - 1.0, _randn(g, n, 3) * (8.0 / n), torch.full(
            (n,), 8.0 / n, dtype=torch.float64, device=g.device)
    if field == "box":           # uniform in [0, 1]^3, one-signed strengths
        return _rand(g, n, 3), _rand(g, n, 3) / n, _rand(g, n) * (2.0 / n)
    th = 2.0 * math.pi * _rand(g, n)
    off = _randn(g, 2, n) * RING_CORE
    rad = RING_R + off[0]
    vol = 2.0 * math.pi * RING_R * 2.0 * math.pi * RING_CORE ** 2 / n
    om = torch.exp(-(off[0] ** 2 + off[1] ** 2) / (2.0 * RING_CORE ** 2)) / (
        2.0 * math.pi * RING_CORE ** 2) * vol
    x = torch.stack([rad * torch.cos(th), rad * torch.sin(th), off[1]], 1)
    a = torch.stack([-torch.sin(th) * om, torch.cos(th) * om, torch.zeros_like(om)], 1)
    return x, a, torch.full((n,), vol, dtype=torch.float64, device=g.device)


def _sigma3(case):
    """Regularisation radius, as the field's workload has it."""
    if case.get("field", "ring") == "ring":
        return RING_SIGMA
    return 0.05


def _soa(x, a, v):
    pv = torch.cat([x, v[:, None]], 1).float().contiguous()
    al = torch.cat([a, torch.zeros_like(a[:, :1])], 1).float().contiguous()
    return pv, al


def _sheet(n, g):
    """2D sheet {x, y, circulation, area} with the areas and circulations
    varying by a tenth (a remeshed sheet's do), FP64 (n, 4)."""
    x = (torch.arange(n, dtype=torch.float64, device=g.device) + 0.5) / n
    y = 0.01 * torch.sin(2.0 * math.pi * x)
    j = _randn(g, 2, n) * 1e-4
    c = (1.0 + 0.1 * _randn(g, n)) / n
    ar = (1.0 + 0.1 * _rand(g, n)) / (float(n) * n)
    return torch.stack([x + j[0], y + j[1], c, ar], 1)


def _lattice(nx, ny, g):
    """Spanwise bound segments of an nx x ny lattice on [0, 4] x [0, 1], as
    {start, strength} and {end, 0} in FP32."""
    dx, dy = 4.0 / nx, 1.0 / ny
    i = torch.arange(nx, device=g.device, dtype=torch.float64).repeat_interleave(ny)
    j = torch.arange(ny, device=g.device, dtype=torch.float64).repeat(nx)
    xq, z = i * dx + dx / 4.0, torch.zeros_like(i)
    s = 1.0 + 0.1 * _randn(g, nx * ny)
    fa = torch.stack([xq, j * dy, z, s], 1).float().contiguous()
    fb = torch.stack([xq, (j + 1.0) * dy, z, z], 1).float().contiguous()
    return fa, fb


def _wake(n, g):
    """Particles in the box [0, 6] x [-0.5, 1.5] x [-0.5, 0.5] around a lattice."""
    u = _rand(g, n, 3)
    x = torch.stack([6.0 * u[:, 0], 2.0 * u[:, 1] - 0.5, u[:, 2] - 0.5], 1)
    return _soa(x, _randn(g, n, 3) * (8.0 / n), torch.full((n,), 8.0 / n, dtype=torch.float64,
                                                           device=g.device))


def _collocation(nx, ny, n, g):
    """Points of a slightly cambered lattice's panels with unit normals."""
    k = torch.arange(n, device=g.device) % (nx * ny)
    i, j = (k // ny).double(), (k % ny).double()
    x = torch.stack([(i + 0.75) * 4.0 / nx, (j + 0.5) / ny, 0.002 * _rand(g, n)], 1)
    t = 0.1 * (_rand(g, n) - 0.5)
    e = torch.stack([torch.sin(t), torch.zeros_like(t), torch.cos(t)], 1)
    pad = torch.zeros_like(t)[:, None]
    return torch.cat([x, pad], 1).float().contiguous(), torch.cat([e, pad], 1).float().contiguous()


def _cloud_inputs(case, g):
    """(offsets, radii, pv, a): sizes log-uniform in [lo, hi] on a fixed grid
    of quantiles (so that every seed costs the same), in a random order."""
    nc = case["n_clouds"]
    q = (np.arange(nc) + 0.5) / nc
    sizes = np.rint(np.exp(math.log(case["lo"]) + q * math.log(case["hi"] / case["lo"]))).astype(np.int64)
    order = torch.randperm(nc, generator=g, device=g.device).cpu().numpy()
    sizes = sizes[order]
    off = np.zeros(nc + 1, np.int64)
    off[1:] = np.cumsum(sizes)
    n = int(off[-1])
    per = torch.from_numpy(np.repeat(sizes, sizes).astype(np.float64)).to(g.device)
    x, a = _rand(g, n, 3), _randn(g, n, 3) / per[:, None]
    sig = (0.01 + 0.09 * _rand(g, nc)).float().cpu().numpy()
    return off, sig, *_soa(x, a, 1.0 / per)


# --------------------------------------------------------------------------
# prepare and run
# --------------------------------------------------------------------------

def _ref(obj):
    return ctypes.cast(ctypes.pointer(obj), ctypes.c_void_p)


def _ptr(a):
    return ctypes.c_void_p(a.ctypes.data)


def _inputs(case, seed, dev):
    """The inputs of a case as tensors (FP32, the library's layouts)."""
    g = _gen(seed, dev)
    kind = case["kind"]
    if kind == "p3d":
        s = _soa(*_points3(case["field"], case["n_src"], g))
        t = s if not case["n_tgt"] else _soa(*_points3(case["field"], case["n_tgt"], g))
        return dict(spv=s[0], sa=s[1], tpv=t[0], ta=t[1])
    if kind == "p2d":
        return dict(s=_sheet(case["n"], g).float().contiguous())
    if kind == "f3d":
        fa, fb = _lattice(case["nx"], case["ny"], g)
        pv, a = _wake(case["n_tgt"], g)
        return dict(fa=fa, fb=fb, tpv=pv, ta=a)
    if kind == "clouds":
        off, sig, pv, a = _cloud_inputs(case, g)
        return dict(off=off, sig=sig, pv=pv, a=a)
    if kind == "relax":
        pv, a = _soa(*_points3("ring", case["n"], g))
        # strengths a little off the field's direction, as after some steps
        a[:, :3] += 0.1 * a[:, :3].norm(dim=1, keepdim=True) * _randn(g, case["n"], 3).float()
        return dict(pv=pv, a=a)
    if kind == "vort":
        spv, sa = _soa(*_points3("ring", case["n_src"], g))
        tpv, _ = _soa(*_points3("ring", case["n_tgt"], g))
        return dict(spv=spv, sa=sa, tpv=tpv)
    if kind == "influence":
        fa, fb = _lattice(case["nx"], case["ny"], g)
        mes, dirs = _collocation(case["nx"], case["ny"], case["n_mes"], g)
        return dict(fa=fa, fb=fb, mes=mes, dir=dirs)
    if kind == "host":
        ns, nt = case["n_src"], case["n_tgt"]
        if case["fn"].startswith("P2D"):
            s, t = _sheet(ns, g), _sheet(nt, g)
            return dict(s=s.float(), t=t.float())
        if case["fn"].startswith("F3D"):
            nx = max(1, int(math.sqrt(ns)))
            fa, fb = _lattice(nx, max(1, ns // nx), g)
            pv, a = _wake(nt, g)
            return dict(fa=fa, fb=fb, tpv=pv, ta=a)
        s, t = _soa(*_points3("box", ns, g)), _soa(*_points3("box", nt, g))
        return dict(spv=s[0], sa=s[1], tpv=t[0], ta=t[1])
    if case["dim"] == 3:
        pv, a = _soa(*_points3("ring", case["n"], g))
        return dict(pv=pv, a=a)
    u = _rand(g, case["n"], 2)   # 2D remeshing: a patch of vorticity
    x = 2.0 * u - 1.0
    om = torch.exp(-8.0 * (x ** 2).sum(1)) * (4.0 / case["n"])
    return dict(s=torch.cat([x, om[:, None], torch.full_like(om, 4.0 / case["n"])[:, None]], 1).float())


def _p3d_records(pv, a):
    pv, a = pv.cpu().numpy(), a.cpu().numpy()
    return make_p3d(pv[:, :3], a[:, :3], pv[:, 3])


def _p2d_records(s):
    s = s.cpu().numpy()
    return make_p2d(s[:, :2], s[:, 2], s[:, 3])


def _f3d_records(fa, fb):
    fa, fb = fa.cpu().numpy(), fb.cpu().numpy()
    return make_f3d(fa[:, :3], fb[:, :3], fa[:, 3])


def prepare(case, seed):
    cv.initialise()
    dev = torch.device("cuda")
    kind = case["kind"]
    i = _inputs(case, seed, dev)
    st = dict(case=case, **i)

    def out(*shape):
        return torch.empty(*shape, dtype=torch.float32, device=dev)

    if kind == "p3d":
        nt = i["tpv"].shape[0]
        o = {k: out(nt, 3) for k in ("vel", "dvort", "visc") if case[k]}
        at = {k: o[k].data_ptr() if k in o else None for k in ("vel", "dvort", "visc")}
        st["prob"] = D.P3DProblem(i["spv"].data_ptr(), i["sa"].data_ptr(), i["spv"].shape[0],
                                  i["tpv"].data_ptr(), i["ta"].data_ptr(), nt, at["vel"],
                                  at["dvort"], at["visc"], REG_ID[case["reg"]], _sigma3(case), NU,
                                  case["acc"])
        st["out"] = o
    elif kind == "p2d":
        n = case["n"]
        o = dict(vel=out(n, 2))
        if case["visc"]:
            o["visc"] = out(n)
        st["prob"] = D.P2DProblem(i["s"].data_ptr(), n, i["s"].data_ptr(), n, o["vel"].data_ptr(),
                                  o["visc"].data_ptr() if case["visc"] else None,
                                  REG_ID[case["reg"]], 4.0 / math.sqrt(n), 1e-4, 1)
        st["out"] = o
    elif kind == "f3d":
        nt = case["n_tgt"]
        o = {k: out(nt, 3) for k in ("vel", "dvort") if case[k]}
        st["prob"] = D.F3DProblem(i["fa"].data_ptr(), i["fb"].data_ptr(), i["fa"].shape[0],
                                  i["tpv"].data_ptr(), i["ta"].data_ptr(), nt,
                                  o["vel"].data_ptr() if case["vel"] else None,
                                  o["dvort"].data_ptr() if case["dvort"] else None, 1)
        st["out"] = o
    elif kind == "clouds":
        n = i["pv"].shape[0]
        st["out"] = dict(vel=out(n, 3), dvort=out(n, 3))
        st["batch"] = D.Batch(i["off"], i["sig"], case["reg"], cv.OUT_VEL | cv.OUT_DVORT, case["acc"])
        st["args"] = [_Gpu(i["pv"]), _Gpu(i["a"]), _Gpu(st["out"]["vel"]), _Gpu(st["out"]["dvort"])]
    elif kind == "relax":
        st["args"] = [_Gpu(i["pv"]), _Gpu(i["a"])]
    elif kind == "vort":
        st["out"] = dict(vort=out(case["n_tgt"], 3))
        st["prob"] = D.VortProblem(i["spv"].data_ptr(), i["sa"].data_ptr(), case["n_src"],
                                   i["tpv"].data_ptr(), case["n_tgt"], st["out"]["vort"].data_ptr(),
                                   REG_ID[case["reg"]], RING_SIGMA, 1)
    elif kind == "influence":
        nf, nm = i["fa"].shape[0], case["n_mes"]
        st["out"] = dict(matrix=out(nm, nf))
        st["args"] = [_Gpu(i["fa"]), _Gpu(i["fb"]), nf, _Gpu(i["mes"]), _Gpu(i["dir"]), nm,
                      _Gpu(st["out"]["matrix"])]
    elif kind == "host":
        st.update(_prepare_host(case, i))
    else:
        st.update(_prepare_remesh(case, i))
    return st


def _prepare_host(case, i):
    """Host records and the arrays of pointers to them that the C API takes."""
    fn, L = case["fn"], cv.lib()
    k = cv.vortfunc(case["reg"])
    st = dict(kfn=k)
    if fn == "P2D_vel":
        src = _p2d_records(i["s"])
        mes = np.ascontiguousarray(i["t"][:, :2].cpu().numpy())
        sig = 4.0 / math.sqrt(case["n_src"])
    elif fn == "F3D_vel":
        src = _f3d_records(i["fa"], i["fb"])
        mes = np.ascontiguousarray(i["tpv"][:, :3].cpu().numpy())
    else:
        src = _p3d_records(i["spv"], i["sa"])
        tgt = _p3d_records(i["tpv"], i["ta"])
        mes = np.ascontiguousarray(tgt["coord"])
        sig = 0.05
    ps, _ = pointer_array(src)
    out = np.zeros_like(mes)
    st.update(src=src, ps=ps, mes=mes, hout=out)
    if fn == "F3D_vel":
        st["call"] = (L.cvtx_F3D_M2M_vel, (_ptr(ps), len(src), _ptr(mes), len(mes), _ptr(out)))
    elif fn in ("P3D_dvort", "P3D_visc"):
        pt, _ = pointer_array(tgt)
        st.update(tgt=tgt, pt=pt)
        head = (_ptr(ps), len(src), _ptr(pt), len(tgt), _ptr(out), _ref(k), sig)
        st["call"] = ((L.cvtx_P3D_M2M_dvort, head) if fn == "P3D_dvort"
                      else (L.cvtx_P3D_M2M_visc_dvort, head + (NU,)))
    else:
        f = {"P3D_vel": L.cvtx_P3D_M2M_vel, "P3D_vort": L.cvtx_P3D_M2M_vort,
             "P2D_vel": L.cvtx_P2D_M2M_vel}[fn]
        st["call"] = (f, (_ptr(ps), len(src), _ptr(mes), len(mes), _ptr(out), _ref(k), sig))
    return st


def _prepare_remesh(case, i):
    L = cv.lib()
    if case["dim"] == 3:
        rec, dt, f = _p3d_records(i["pv"], i["a"]), P3D_DTYPE, L.cvtx_P3D_redistribute_on_grid
    else:
        rec, dt, f = _p2d_records(i["s"]), P2D_DTYPE, L.cvtx_P2D_redistribute_on_grid
    ps, _ = pointer_array(rec)
    cap = max(4096, 2 * case["n"])   # room for the new particles, kept from step to step
    buf = np.zeros(cap, dt)
    r = cv.redistfunc(case["fn"])
    return dict(src=rec, ps=ps, buf=buf, rf=r,
                call=(f, (_ptr(ps), len(rec), _ptr(buf), cap, _ref(r), case["h"], 0.01)))


def run(st):
    kind = st["case"]["kind"]
    if kind == "p3d":
        D.p3d_eval(st["prob"])
    elif kind == "p2d":
        D.p2d_eval(st["prob"])
    elif kind == "f3d":
        D.f3d_eval(st["prob"])
    elif kind == "clouds":
        st["batch"].eval(*st["args"])
    elif kind == "relax":
        D.relax_eval(*st["args"], st["case"]["n"], FDT, st["case"]["reg"], RING_SIGMA)
        return st["a"]
    elif kind == "vort":
        D.vort_eval(st["prob"])
    elif kind == "influence":
        D.f3d_inf_eval(*st["args"])
    elif kind == "host":
        f, args = st["call"]
        f(*args)
        return st["hout"]
    else:
        f, args = st["call"]
        n = f(*args)
        if n < 0:
            raise RuntimeError("remeshing failed: " + cv.last_error())
        # the caller's whole array: its first n records are the new particles
        return dict(n=n, **{k: st["buf"][k] for k in st["buf"].dtype.names})
    return st["out"]


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------

# operations per pair: add, multiply, compare, select and transcendental one
# each, a fused multiply-add two
_F3 = {"singular": (28, 24, 4), "winckelmans": (31, 26, 16), "planetary": (30, 26, 4),
       "gaussian": (48, 31, 15)}
_F2 = {"singular": (13, 0), "winckelmans": (15, 6), "planetary": (14, 0), "gaussian": (16, 5)}


def work(case):
    kind = case["kind"]
    if kind == "p3d":
        ns, nt = case["n_src"], case["n_tgt"] or case["n_src"]
        v, d, s = _F3[case["reg"]]
        f = v + (d if case["dvort"] else 0) + (s if case["visc"] else 0)
        outs = sum(case[k] for k in ("vel", "dvort", "visc"))
        return dict(bytes=32.0 * ns + (32.0 * nt if case["n_tgt"] else 0.0) + 12.0 * nt * outs,
                    flops=float(f) * ns * nt)
    if kind == "p2d":
        n = case["n"]
        v, s = _F2[case["reg"]]
        return dict(bytes=16.0 * n + (12.0 if case["visc"] else 8.0) * n,
                    flops=float(v + (s if case["visc"] else 0)) * n * n)
    if kind == "f3d":
        nf, nt = case["nx"] * case["ny"], case["n_tgt"]
        f = 100 if case["vel"] and case["dvort"] else (56 if case["vel"] else 76)
        return dict(bytes=32.0 * nf + 32.0 * nt + 12.0 * nt * (case["vel"] + case["dvort"]),
                    flops=float(f) * nf * nt)
    if kind == "clouds":
        q = (np.arange(case["n_clouds"]) + 0.5) / case["n_clouds"]
        s = np.exp(math.log(case["lo"]) + q * math.log(case["hi"] / case["lo"]))
        v, d, _ = _F3[case["reg"]]
        return dict(bytes=56.0 * float(s.sum()), flops=float(v + d) * float((s * s).sum()))
    if kind in ("relax", "vort"):
        ns = case["n"] if kind == "relax" else case["n_src"]
        nt = case["n"] if kind == "relax" else case["n_tgt"]
        c = 5.0 * RING_SIGMA   # pairs inside the cut-off box, along and across the core
        share = c / (math.pi * RING_R) * math.erf(c / (2.0 * RING_CORE)) ** 2
        return dict(bytes=32.0 * ns + 28.0 * nt, flops=23.0 * share * ns * nt)
    if kind == "influence":
        nf, nm = case["nx"] * case["ny"], case["n_mes"]
        return dict(bytes=4.0 * nf * nm + 32.0 * (nf + nm), flops=47.0 * nf * nm)
    ns = case.get("n_src", case.get("n"))
    if kind == "host":
        nt = case["n_tgt"]
        f = {"P3D_vel": 31, "P3D_dvort": 51, "P3D_visc": 25, "P2D_vel": 15, "F3D_vel": 56,
             "P3D_vort": 23}[case["fn"]]
        return dict(bytes=28.0 * ns + 24.0 * nt, flops=float(f) * ns * nt)
    w = (5 if case["fn"] in ("m4p", "lambda3", "lambda2") else 3) ** case["dim"]
    rec = 28.0 if case["dim"] == 3 else 16.0
    return dict(bytes=rec * ns, flops=8.0 * w * ns)


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------

# pairs that are summed again in 64 bits (a few seconds' worth)
_MOST = {"p2d": 1.0e11, "f3d": 2.0e10, "relax": 4.0e10, "vort": 4.0e10}
_S2PI = math.sqrt(2.0 / math.pi)


def _reg3(reg, q):
    """(G, H, eta) at q = rho^2: G = g / rho^3, H = (3 G - zeta) / rho^2."""
    if reg == "singular":
        y = q.rsqrt()
        g = y * y * y
        return g, 3.0 * g * y * y, None
    if reg == "winckelmans":
        y2 = 1.0 / (q + 1.0)
        y = y2.sqrt()
        y5 = y2 * y2 * y
        return (q + 2.5) * y5, 3.0 * (q + 3.5) * y5 * y2, 52.5 * y5 * y2 * y2
    if reg == "planetary":
        y = q.rsqrt()
        g = y * y * y
        inside = q < 1.0
        return torch.where(inside, torch.ones_like(g), g), torch.where(
            inside, torch.zeros_like(g), 3.0 * g * y * y), None
    z = _S2PI * torch.exp(-0.5 * q)
    rho = q.sqrt()
    g = (torch.erf(rho * math.sqrt(0.5)) - rho * z) / (q * rho)
    h = (3.0 * g - z) / q
    sg, sh, c = torch.zeros_like(q), torch.zeros_like(q), 1.0
    for k in range(12, -1, -1):
        c = _S2PI * (-0.5) ** k / math.factorial(k)
        sg = sg * q + c / (2 * k + 3)
    for k in range(12, 0, -1):
        c = _S2PI * (-0.5) ** k / math.factorial(k)
        sh = sh * q + c * (3.0 / (2 * k + 3) - 1.0)
    small = q < 0.5
    return torch.where(small, sg, g), torch.where(small, sh, h), z


def _chunks(nt, ns, most=6.0e6):
    step = max(1, int(most / max(1, ns)))
    for a in range(0, nt, step):
        yield a, min(nt, a + step)


def _exact_p3d(s, sa, sv, t, ta, tv, reg, sigma, nu, want):
    sg = float(np.float32(sigma))
    k4 = 1.0 / (4.0 * math.pi)
    length = 1.0 if reg == "singular" else abs(sg)
    nt = t.shape[0]
    o = {k: torch.empty(nt, 3, dtype=torch.float64, device=t.device) for k in want}
    for a, b in _chunks(nt, s.shape[0]):
        dx, dy, dz = (t[a:b, None, c] - s[None, :, c] for c in range(3))
        r2 = dx * dx + dy * dy + dz * dz
        zero = r2 == 0.0
        g, h, eta = _reg3(reg, torch.where(zero, torch.ones_like(r2), r2) / length ** 2)
        g = torch.where(zero, torch.zeros_like(g), g) / length ** 3
        if "vel" in want or "dvort" in want:
            cx = dy * sa[:, 2] - dz * sa[:, 1]
            cy = dz * sa[:, 0] - dx * sa[:, 2]
            cz = dx * sa[:, 1] - dy * sa[:, 0]
        if "vel" in want:
            o["vel"][a:b] = -k4 * torch.stack([(g * c).sum(1) for c in (cx, cy, cz)], 1)
        if "dvort" in want:
            h = torch.where(zero, torch.zeros_like(h), h) / length ** 5
            at = ta[a:b]
            w = h * (at[:, None, 0] * cx + at[:, None, 1] * cy + at[:, None, 2] * cz)
            grad = torch.stack([(w * d).sum(1) for d in (dx, dy, dz)], 1)
            o["dvort"][a:b] = math.copysign(k4, sg) * (torch.linalg.cross(at, g @ sa) + grad)
        if "visc" in want:
            eta = torch.where(zero, torch.zeros_like(eta), eta)
            o["visc"][a:b] = 2.0 * nu / sg ** 2 * (tv[a:b, None] * (eta @ sa)
                                                   - ta[a:b] * (eta @ sv)[:, None])
    return o


def _exact_p2d(s, t, reg, sigma, nu, visc):
    sg = float(np.float32(sigma))
    nt = t.shape[0]
    vel = torch.empty(nt, 2, dtype=torch.float64, device=t.device)
    vs = torch.empty(nt, dtype=torch.float64, device=t.device)
    for a, b in _chunks(nt, s.shape[0]):
        dx, dy = t[a:b, None, 0] - s[None, :, 0], t[a:b, None, 1] - s[None, :, 1]
        r2 = dx * dx + dy * dy
        zero = r2 == 0.0
        r2 = torch.where(zero, torch.ones_like(r2), r2)
        q = r2 / sg ** 2
        if reg == "singular":
            k = 1.0 / r2
        elif reg == "planetary":
            k = 1.0 / torch.clamp(r2, min=sg ** 2)
        elif reg == "winckelmans":
            k = (q + 2.0) / (q + 1.0) ** 2 / sg ** 2
            eta = 24.0 * torch.exp(4.0 / (q + 1.0) ** 3) / (q + 1.0) ** 4
        else:
            k = -torch.expm1(-0.5 * q) / r2
            eta = torch.exp(-0.5 * q)
        k = torch.where(zero, torch.zeros_like(k), k) * s[:, 2]
        vel[a:b, 0] = (k * dy).sum(1) / (2.0 * math.pi)
        vel[a:b, 1] = -(k * dx).sum(1) / (2.0 * math.pi)
        if visc:
            e = torch.where(zero, torch.zeros_like(eta), eta)
            x = t[a:b, None, 3] * s[:, 2] - t[a:b, None, 2] * s[:, 3]
            vs[a:b] = 2.0 * nu / sg ** 2 * (e * x).sum(1)
    return dict(vel=vel, visc=vs) if visc else dict(vel=vel)


def _exact_f3d(fa, fb, t, ta, want, dirs=None):
    nt = t.shape[0]
    o = {k: torch.empty(nt, 3, dtype=torch.float64, device=t.device) for k in want}
    if dirs is not None:
        o = dict(matrix=torch.empty(nt, fa.shape[0], dtype=torch.float64, device=t.device))
    r0 = fb[:, :3] - fa[:, :3]
    g = fa[:, 3] / (4.0 * math.pi)
    length = r0.norm(dim=1)
    for a, b in _chunks(nt, fa.shape[0]):
        p = [t[a:b, None, c] - fa[None, :, c] for c in range(3)]
        q = [t[a:b, None, c] - fb[None, :, c] for c in range(3)]
        c = [p[1] * q[2] - p[2] * q[1], p[2] * q[0] - p[0] * q[2], p[0] * q[1] - p[1] * q[0]]
        cc = c[0] ** 2 + c[1] ** 2 + c[2] ** 2
        n1 = (p[0] ** 2 + p[1] ** 2 + p[2] ** 2).sqrt()
        n2 = (q[0] ** 2 + q[1] ** 2 + q[2] ** 2).sqrt()
        d = p[0] * q[0] + p[1] * q[1] + p[2] * q[2]
        n12 = n1 * n2
        k = g * (n1 + n2) / n12 * torch.where(d >= 0.0, 1.0 / (n12 + d), (n12 - d) / cc)
        k = torch.where(torch.isfinite(k), k, torch.zeros_like(k))
        if dirs is not None:
            e = dirs[a:b]
            o["matrix"][a:b] = k * (c[0] * e[:, None, 0] + c[1] * e[:, None, 1] + c[2] * e[:, None, 2])
            continue
        if "vel" in want:
            o["vel"][a:b] = torch.stack([(k * x).sum(1) for x in c], 1)
        if "dvort" in want:
            p12 = sum(r0[:, i] * (p[i] + q[i]) for i in range(3))
            w = -3.0 * g / length * cc.sqrt() * p12 / (n12 * (n1 + n2))
            ok = (cc > 0.0) & torch.isfinite(w)
            w = torch.where(ok, w, torch.zeros_like(w)).sum(1)
            s = torch.where(ok, k, torch.zeros_like(k)) @ r0
            at = ta[a:b]
            o["dvort"][a:b] = at * w[:, None] - torch.linalg.cross(s, at)
    return o


def _exact_vort(s, sa, t, reg, sigma):
    """Vorticity with the reference's FP32 cut-off box: s, t FP32, sums FP64."""
    sg = float(np.float32(sigma))
    cut = float(np.float32(5.0) * np.float32(sigma))
    k = 7.5 if reg == "winckelmans" else _S2PI
    o = torch.empty(t.shape[0], 3, dtype=torch.float64, device=t.device)
    sd, td = s.double(), t.double()
    for a, b in _chunks(t.shape[0], s.shape[0]):
        inside = None
        r2 = 0.0
        for c in range(3):
            w = (s[None, :, c] - t[a:b, None, c]).abs() < cut
            inside = w if inside is None else inside & w
            r2 = r2 + (sd[None, :, c] - td[a:b, None, c]) ** 2
        q = r2 / sg ** 2
        z = (q + 1.0) ** -3.5 if reg == "winckelmans" else torch.exp(-0.5 * q)
        o[a:b] = torch.where(inside, z, torch.zeros_like(z)) @ sa
    return o * (k / (4.0 * math.pi * sg ** 3))


def exact(case, seed):
    kind = case["kind"]
    if kind == "remesh":
        return None   # which nodes there are follows from FP32 arithmetic
    w = work(case)
    ns = case.get("n_src") or case.get("n") or case.get("nx", 0) * case.get("ny", 0)
    nt = case.get("n_tgt") or case.get("n_mes") or ns
    pairs = w["flops"] / 57.0 if kind == "clouds" else float(ns) * nt
    if pairs > _MOST.get(kind, 1.5e10):
        return None
    i = _inputs(case, seed, torch.device("cuda"))
    x = {k: v.double() if isinstance(v, torch.Tensor) else v for k, v in i.items()}
    if kind == "p3d":
        want = [k for k in ("vel", "dvort", "visc") if case[k]]
        return _exact_p3d(x["spv"][:, :3], x["sa"][:, :3], x["spv"][:, 3], x["tpv"][:, :3],
                          x["ta"][:, :3], x["tpv"][:, 3], case["reg"], _sigma3(case),
                          float(np.float32(NU)), want)
    if kind == "p2d":
        return _exact_p2d(x["s"], x["s"], case["reg"], 4.0 / math.sqrt(case["n"]),
                          float(np.float32(1e-4)), case["visc"])
    if kind == "f3d":
        return _exact_f3d(x["fa"], x["fb"], x["tpv"], x["ta"][:, :3],
                          [k for k in ("vel", "dvort") if case[k]])
    if kind == "clouds":
        off, o = i["off"], []
        for c in range(case["n_clouds"]):
            p, a = x["pv"][off[c]:off[c + 1]], x["a"][off[c]:off[c + 1], :3]
            o.append(_exact_p3d(p[:, :3], a, p[:, 3], p[:, :3], a, p[:, 3], case["reg"],
                                i["sig"][c], 0.0, ["vel", "dvort"]))
        return {k: torch.cat([y[k] for y in o]) for k in ("vel", "dvort")}
    if kind == "relax":
        om = _exact_vort(i["pv"], x["a"][:, :3], i["pv"], case["reg"], RING_SIGMA)
        a, f = x["a"].clone(), float(np.float32(FDT))
        r = a[:, :3].norm(dim=1) / om.norm(dim=1)
        a[:, :3] = a[:, :3] * (1.0 - f) + om * (r * f)[:, None]
        return a
    if kind == "vort":
        return dict(vort=_exact_vort(i["spv"], x["sa"][:, :3], i["tpv"], case["reg"], RING_SIGMA))
    if kind == "influence":
        return _exact_f3d(x["fa"], x["fb"], x["mes"], None, [], dirs=x["dir"])
    if case["fn"] == "P2D_vel":
        return _exact_p2d(x["s"], x["t"], case["reg"], 4.0 / math.sqrt(case["n_src"]), 0.0,
                          False)["vel"].cpu().numpy()
    if case["fn"] == "F3D_vel":
        return _exact_f3d(x["fa"], x["fb"], x["tpv"], None, ["vel"])["vel"].cpu().numpy()
    if case["fn"] == "P3D_vort":
        return _exact_vort(i["spv"], x["sa"][:, :3], i["tpv"], case["reg"], 0.05).cpu().numpy()
    k = case["fn"][4:]
    return _exact_p3d(x["spv"][:, :3], x["sa"][:, :3], x["spv"][:, 3], x["tpv"][:, :3],
                      x["ta"][:, :3], x["tpv"][:, 3], case["reg"], 0.05, float(np.float32(NU)),
                      [k])[k].cpu().numpy()
