"""Timed cases of the Fluid2d timestep path, through its public entry points.

Each case is one pass of work as a user's program makes it: steps of a
model on the batched engine, ``Fluid2d.loop``, a multigrid solve through
``Gmg``, or a run of the kernel-level routines.  ``prepare`` builds what such
a program holds before the call (inputs from the seed, the engine or solver
handle), ``run`` makes one pass and returns the arrays it computes, ``work``
counts what a pass cannot do without, and ``exact`` restates a pass in plain
torch FP64.

Kinds of case:

* ``steps``: ``Batch.step`` on one or more instances, dt adapted on the
  device (CFL 0.8, what ``Fluid2d.loop`` does by default);
* ``loop``: ``Fluid2d.loop``, the reference's own driver, which reads the
  diagnostics back after each step;
* ``solve``, ``twov``: ``Gmg.solve`` and ``Gmg.twoVcycle`` on a caller's
  arrays (the two inversions of the time step);
* ``rhs``, ``mg``, ``diag``: the kernel-level routines a right-hand side, one
  multigrid level visit and one set of diagnostics call, in their order.
"""
import math

import numpy as np
import torch

import fluid2d_amd as F
from fluid2d_amd import kernels as K
from fluid2d_amd import workloads
from fluid2d_amd.batch import Batch

NH = 3
CFL = 0.8
OMEGA = 8.0 / 9.0


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest configuration: launches and latency
        dict(name="step-euler-perio-128", kind="steps", model="euler", nx=128, ny=128,
             geometry="perio", precision="fp64", count=1, order=5, steps=8),
        # the headline configuration, plain FP64
        dict(name="step-euler-closed-1024", kind="steps", model="euler", nx=1024, ny=1024,
             geometry="closed", precision="fp64", count=1, order=5, steps=4),
        # the Boussinesq configuration: two tracers, diffusion, 2:1 channel
        dict(name="step-bous-channel-2048x1024", kind="steps", model="boussinesq", nx=2048,
             ny=1024, geometry="xchannel", precision="fp64", count=1, order=5, steps=4),
        # a grid the tiles do not divide, coarsest level 6 x 3, mixed precision
        dict(name="step-bous-channel-384x192-mixed", kind="steps", model="boussinesq", nx=384,
             ny=192, geometry="xchannel", precision="mixed", count=1, order=5, steps=8),
        # an ensemble: sizes 64..512, periodic and closed, in one batch
        dict(name="ensemble-32-mixed", kind="steps", model="euler", nx=0, ny=0, geometry="",
             precision="mixed", count=32, order=5, steps=2),
        # a serving pool of one class in FP64
        dict(name="pool-8-euler-closed-256", kind="steps", model="euler", nx=256, ny=256,
             geometry="closed", precision="fp64", count=8, order=5, steps=4),
        # the reference's driver on its default geometry, host in the loop
        dict(name="loop-euler-disc-256", kind="loop", model="euler", nx=256, ny=256,
             geometry="disc", order=5, steps=8),
        # the drop-in solver: the full inversion and the fast one
        dict(name="gmg-solve-closed-512", kind="solve", nx=512, ny=512, geometry="closed"),
        dict(name="gmg-twov-channel-1024x512", kind="twov", nx=1024, ny=512,
             geometry="xchannel"),
        # the kernel-level routines: a right-hand side on a small grid, a
        # level visit of a large one, the diagnostics of a large one
        dict(name="kernels-rhs-256", kind="rhs", nx=256, ny=256, geometry="closed", order=5),
        dict(name="kernels-mg-2048", kind="mg", nx=2048, ny=2048, geometry="closed"),
        dict(name="kernels-diag-2048x1024", kind="diag", nx=2048, ny=1024,
             geometry="xchannel"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A grid side lo..hi that halves down to 4 or 3 (the coarsest level)."""
    while True:
        s = rng.choice((1, 1, 3)) << rng.randrange(3, 12)
        if lo <= s <= hi:
            return s


def _width(rng, ny):
    # 3:2 halves down with powers of two only
    return ny * rng.choice((2, 2, 4, 4 if ny % 3 == 0 else 3)) // 2


def draw(rng):
    kind = rng.choice(("steps", "steps", "steps", "loop", "solve", "twov", "rhs", "mg", "diag"))
    geometry = rng.choice(("perio", "closed", "xchannel", "disc"))
    c = dict(kind=kind, geometry=geometry)
    if kind in ("steps", "loop"):
        c["model"] = rng.choice(("euler", "euler", "boussinesq"))
        big = c["model"] == "boussinesq"
        c["order"] = rng.choice((5, 5, 5, 3, 4))
        c["steps"] = rng.choice((2, 4, 8))
        ny = _size(rng, 64, 512)
        c.update(nx=_width(rng, ny), ny=ny)
        if geometry == "disc" or big and geometry == "perio":
            c["geometry"] = "closed" if big else geometry
        if kind == "steps":
            c["precision"] = rng.choice(("fp64", "fp64", "mixed"))
            c["count"] = rng.choice((1, 1, 2, 4)) if ny <= 256 else 1
        return c
    if kind in ("solve", "twov"):
        ny = _size(rng, 64, 512)
        c.update(nx=_width(rng, ny), ny=ny)
        return c
    if kind == "rhs":
        c["order"] = rng.choice((5, 5, 3, 1, 2, 4, 6))
    if kind == "mg":  # two levels of a multigrid: even sides
        c.update(nx=2 * _log_int(rng, 32, 1024), ny=2 * _log_int(rng, 32, 1024))
    else:
        c.update(nx=_log_int(rng, 64, 2048), ny=_log_int(rng, 64, 1024))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _View:
    """A device array of the library as torch sees it; holds the array's
    owner for as long as a tensor on it lives."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8",
                                         "data": (int(ptr), False), "strides": None,
                                         "version": 3}


def _view(ptr, shape, owner):
    return torch.as_tensor(_View(ptr, shape, owner), device="cuda")


def _param(case, model, nx, ny, geometry):
    kw = dict(modelname=model, nx=nx, ny=ny, Lx=nx / ny, Ly=1.0, geometry=geometry,
              order=case["order"], cfl=CFL, flux_splitting_method="parabolic",
              timestepping="RK3_SSP", autotune=False)
    if model == "boussinesq":
        kw.update(diffusion=True, Kdiff=1e-5, gravity=1.0)
    return F.Param(**kw)


def _dtmax(g, model):
    # the buoyancy velocity scale, 1, bounds the steps of a stratified flow
    return CFL * min(g.dx, g.dy) if model == "boussinesq" else 5.0


def _instances(case, seed):
    """(param, grid, initial fields) of each instance of a steps/loop case."""
    out = []
    if case["nx"] == 0:
        specs = workloads.ensemble_specs(case["count"], seed=4)
    else:
        specs = [(None, None)] * case["count"]
    for k, (kw, _) in enumerate(specs):
        if kw is None:
            p = _param(case, case["model"], case["nx"], case["ny"], case["geometry"])
        else:
            p = _param(case, "euler", kw["nx"], kw["ny"], kw["geometry"])
        g = F.Grid(p)
        s = 1000 * (seed % 1000003) + k
        if p.modelname == "euler":
            f = {"vorticity": workloads.turbulence(g, s)}
        else:  # an overturning already under way: every field has structure
            f = {"vorticity": workloads.turbulence(g, s),
                 "buoyancy": workloads.rayleigh_taylor(g, s)
                 + 0.1 * workloads.turbulence(g, s + 500009)}
        out.append((p, g, f))
    return out


def _mask(nx, ny, geometry):
    """int8 cell mask and corner mask of a geometry, with halo."""
    g = F.Grid(F.Param(nx=nx, ny=ny, Lx=nx / ny, Ly=1.0, geometry=geometry))
    m = g.msk
    mskp = np.zeros_like(m)
    mskp[:-1, :-1] = (m[:-1, :-1] + m[:-1, 1:] + m[1:, :-1] + m[1:, 1:]) == 4
    return g, m, mskp


def _fields(seed, n, m1, n1, dev):
    """n smooth random fields of shape (m1, n1) with a periodic halo: a
    k^-1 spectrum, as the turbulence of the time steps has."""
    gen = torch.Generator(device="cpu").manual_seed(int(seed) % (1 << 62))
    ny, nx = m1 - 2 * NH, n1 - 2 * NH
    out = []
    for _ in range(n):
        z = torch.randn(ny, nx, generator=gen, dtype=torch.float64).to(dev)
        k = torch.sqrt(torch.fft.fftfreq(ny, 1.0 / ny, device=dev, dtype=torch.float64)[:, None] ** 2
                       + torch.fft.fftfreq(nx, 1.0 / nx, device=dev, dtype=torch.float64)[None] ** 2)
        z = torch.fft.ifft2(torch.fft.fft2(z) / (1.0 + k)).real
        a = torch.zeros(m1, n1, dtype=torch.float64, device=dev)
        a[NH:-NH, NH:-NH] = z / z.std()
        out.append(_fill(a))
    return out


def _mg_inputs(case, seed, dev):
    g, _, mskp = _mask(case["nx"], case["ny"], case["geometry"])
    if case["kind"] == "mg":
        lev = _levels(torch.from_numpy(mskp).to(dev), g.dx, g.dy, 2)
    else:
        lev = None
    x, b = _fields(seed, 2, g.nyl, g.nxl, dev)
    mk = torch.from_numpy(mskp).to(dev)
    return g, mskp, lev, 1e-3 * x * mk, _fill(b * mk)


def _rhs_inputs(case, seed, dev):
    g, msk, _ = _mask(case["nx"], case["ny"], case["geometry"])
    # with means of their own, so that no sum of theirs is rounding alone
    w, b, psi = (f + c for f, c in zip(_fields(seed, 3, g.nyl, g.nxl, dev), (0.25, 0.5, 1.0)))
    mk = torch.from_numpy(msk).to(dev)
    u, v = torch.zeros_like(w), torch.zeros_like(w)
    _ortho(mk, 0.05 * psi, g.dx, g.dy, u, v)
    umax = float((u.abs() + v.abs()).max())
    cst = [g.dx, g.dy, 0.05, umax, 0.05 if case.get("order", 5) % 2 else 0.0]
    return g, mk, _fill(w * mk), _fill(b * mk), psi * mk, u, v, cst


def prepare(case, seed):
    kind = case["kind"]
    if kind == "steps":
        inst = _instances(case, seed)
        # launch shapes as the autotuner picks them: tall tiles for many
        # instances, about 1024 workgroups a phase for one
        cells = sum(g.nx * g.ny for _, g, _ in inst)
        tune = dict(coarse_lds_budget=0, coarse_wave_cells=0,
                    min_tiles=0 if len(inst) > 4 else (4096 if cells > 2000000 else 1024))
        b = Batch([(p, g) for p, g, _ in inst], precision=case["precision"], tuning=tune)
        p0, g0, _ = inst[0]
        b.set_adaptive(True, CFL, _dtmax(g0, p0.modelname))
        b.set_dt(_dtmax(g0, p0.modelname))
        outs = []
        for i, (p, g, f) in enumerate(inst):
            for name, a in f.items():
                b.set_field(i, name, a)
            ptr = F._lib.C.c_void_p()
            F.load().f2d_batch_state_ptr(F._lib.C.c_void_p(b._h), i, F._lib.C.byref(ptr))
            outs.append(_view(ptr.value, (len(b.varnames[i]), g.nyl, g.nxl), b))
        b.set_psi_from_vorticity()
        return {"case": case, "batch": b, "outs": outs}
    if kind == "loop":
        p, g, f = _instances(dict(case, count=1), seed)[0]
        p.dtmax = p.dt = _dtmax(g, p.modelname)
        p.exacthistime, p.freq_his, p.freq_diag = False, 1e30, 1e30
        f2d = F.Fluid2d(p, g)
        for name, a in f.items():
            f2d.model.var.get(name)[...] = a
        f2d.model.set_psi_from_vorticity()
        return {"case": case, "f2d": f2d,
                "out": _view(f2d.model.var.dev.ptr, f2d.model.var.dev.shape, f2d)}
    if kind in ("solve", "twov"):
        g, mskp, _, x, b = _mg_inputs(case, seed, "cuda")
        gmg = F.Gmg(dict(n=g.nx, m=g.ny, nh=NH, dx=g.dx, dy=g.dy, omega=OMEGA), mskp)
        return {"case": case, "gmg": gmg, "x": x, "b": b}
    if kind == "mg":
        _, _, lev, x, b = _mg_inputs(case, seed, "cuda")
        z = torch.zeros_like
        return {"case": case, "msk": lev[0][0], "A": lev[0][1][:5].contiguous(), "msk2": lev[1][0],
                "x": x, "b": b, "r": z(x), "work": z(x), "b2": z(lev[1][1][0])}
    g, mk, w, b, psi, u, v, cst = _rhs_inputs(case, seed, "cuda")
    z = torch.zeros_like
    return {"case": case, "grid": g, "msk": mk, "w": w, "b": b, "psi": psi, "u": u, "v": v,
            "cst": cst, "dw": z(w), "db": z(w), "c": z(w), "du": z(w), "dv": z(w)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "steps":
        s["batch"].step(case["steps"])
        return s["outs"]
    if kind == "loop":
        s["f2d"].loop(nsteps=case["steps"])
        d = s["f2d"].model.diags
        return {"state": s["out"], "diags": [d["maxspeed"], d["ke"], d["enstrophy"]]}
    if kind == "solve":
        x = s["x"].clone()
        _, res = s["gmg"].solve(x, s["b"])
        return {"x": x, "res": res}
    if kind == "twov":
        x = s["x"].clone()
        s["gmg"].twoVcycle(x, s["b"])
        return {"x": x}
    if kind == "mg":
        # one visit of a level on the way down and back up: smooth, residual,
        # restrict; interpolate (the restricted field stands for the coarse
        # solution) and smooth
        x = s["x"].clone()
        K.smoothtwicewitha_fill(s["msk"], s["A"], x, s["b"], OMEGA, s["work"])
        K.computeresidualwitha_fill(s["msk"], s["A"], x, s["b"], s["r"])
        K.restrict_fill(s["msk2"], s["r"], NH, s["b2"])
        K.interpolate(s["msk"], s["msk2"], s["b2"], NH, x, accumulate=True)
        K.smoothtwicewitha_fill(s["msk"], s["A"], x, s["b"], OMEGA, s["work"])
        return {"x": x, "r": s["r"], "b2": s["b2"]}
    g, mk, cst = s["grid"], s["msk"], s["cst"]
    if kind == "rhs":
        adv = K.adv_upwind if case["order"] % 2 else K.adv_centered
        for q, dq in ((s["w"], s["dw"]), (s["b"], s["db"])):
            adv(mk, q, dq, s["u"], s["v"], cst, NH, 1, case["order"])
            K.fillhalo(dq, NH)
        K.add_torque_fill(mk, s["b"], g.dx, NH, 1.0, s["dw"])
        K.add_diffusion_fill(mk, s["w"], g.dx, NH, 1e-5, s["dw"])
        K.add_diffusion_fill(mk, s["b"], g.dx, NH, 1e-5, s["db"])
        K.celltocorner(s["dw"], s["c"])
        K.computeorthogradient(mk, s["psi"], g.dx, g.dy, NH, s["du"], s["dv"])
        return [s["dw"], s["db"], s["c"], s["du"], s["dv"]]
    ke, maxu = K.computekemaxu(mk, s["u"], s["v"], NH)
    z, z2 = K.computesumandnorm(mk, s["w"], NH)
    return [ke, maxu, z, z2, K.computenorm(mk, s["w"], NH),
            K.computedotprod(mk, s["w"], s["b"], NH), K.computesum(mk, s["b"], NH),
            K.domain_integration(s["psi"])]


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: the arrays a pass takes in and those it gives back, once each
    (per step for the time steps).  Flops: of the method, per cell.  A
    V-cycle costs 105 flops per cell of a level (two double sweeps at 80, the
    residual 18, the transfers 7) and the levels add up to 4/3; an F-cycle
    is V-cycles from every level."""
    kind = case["kind"]
    vcyc = 105.0 * 4.0 / 3.0
    fcyc = vcyc * 4.0 / 3.0 + 20.0
    if kind in ("steps", "loop"):
        if case["nx"] == 0:
            cells = sum(kw["nx"] * kw["ny"] for kw, _ in
                        workloads.ensemble_specs(case["count"], seed=4))
        else:
            cells = case["nx"] * case["ny"] * case.get("count", 1)
        euler = case["model"] == "euler"
        # Euler: 3 advections, 2 fast inversions, a full solve of 4 F-cycles;
        # Boussinesq: 6 advections, 3 fast inversions
        fl = 3 * 60 + 4 * vcyc + 4 * fcyc + 60 if euler else 6 * 60 + 6 * vcyc + 60
        nvar = 5 if euler else 6
        return {"bytes": case["steps"] * 2.0 * nvar * 8 * cells,
                "flops": case["steps"] * fl * cells}
    cells = float(case["nx"] * case["ny"])
    if kind == "solve":
        return {"bytes": 3 * 8 * cells, "flops": (4 * (fcyc + 20) + 20) * cells}
    if kind == "twov":
        return {"bytes": 3 * 8 * cells, "flops": 2 * vcyc * cells}
    if kind == "mg":  # msk, five planes of A, x, b in; x, r, b2 out
        return {"bytes": (1.25 + (5 + 2 + 2.25) * 8) * cells, "flops": 108 * cells}
    if kind == "rhs":  # msk, w, b, psi, u, v in; dw, db, c, du, dv out
        return {"bytes": (1 + 10 * 8) * cells, "flops": 160 * cells}
    return {"bytes": (1 + 5 * 8) * cells, "flops": 25 * cells}  # msk, u, v, w, b, psi


# ---------------------------------------------------------------------------
# the same in plain torch FP64: fields (m, n) with a 3-cell halo, masks int8
# ---------------------------------------------------------------------------
def _fill(a):
    m, n = a.shape[-2:]
    a[..., :NH, :] = a[..., m - 2 * NH:m - NH, :].clone()
    a[..., m - NH:, :] = a[..., NH:2 * NH, :].clone()
    a[..., :, :NH] = a[..., :, n - 2 * NH:n - NH].clone()
    a[..., :, n - NH:] = a[..., :, NH:2 * NH].clone()
    return a


def _at(a, lo, hi, dj=0, di=0):
    """a on rows [lo, m - hi) x cols [lo, n - hi), shifted by (dj, di)."""
    m, n = a.shape[-2:]
    return a[..., lo + dj:m - hi + dj, lo + di:n - hi + di]


def _odd(a, dj, di, step=2):
    """Fine values around the points under each interior coarse cell."""
    m, n = a.shape[-2:]
    return a[..., 2 * NH - 2 + dj:m - 2 * NH + 3 + dj + 1:step,
             2 * NH - 2 + di:n - 2 * NH + 3 + di + 1:step]


def _full_weight(a, mc, nc):
    def f(dj, di):
        return _odd(a, dj, di)[..., :mc - 2 * NH, :nc - 2 * NH]
    return (0.25 * f(0, 0) + 0.125 * (f(0, -1) + f(0, 1) + f(-1, 0) + f(1, 0))
            + 0.0625 * (f(-1, -1) + f(-1, 1) + f(1, -1) + f(1, 1)))


def _levels(mskp, dx, dy, most=99):
    """[(mask, 9 operator planes)] from the finest level down."""
    m, n = mskp.shape
    if dx == dy:
        st = [0.25, 0.5, 0.25, 0.5, -3.0, 0.5, 0.25, 0.5, 0.25]
    else:
        bx, by = dy / dx, dx / dy
        st = [0.0, by, 0.0, bx, -2 * (bx + by), bx, 0.0, by, 0.0]
    mf = mskp.double()
    A = torch.zeros(9, m, n, dtype=torch.float64, device=mskp.device)
    for k in range(9):
        _at(A[k], NH, NH)[...] = (st[k] / (dx * dy) * _at(mf, NH, NH, k // 3 - 1, k % 3 - 1)
                                  * _at(mf, NH, NH))
    out = [(mskp, _fill(A))]
    cw = [0.25, 0.5, 0.25]
    while len(out) < most and min(m, n) - 2 * NH > 4:
        mc, nc = (m - 2 * NH) // 2 + 2 * NH, (n - 2 * NH) // 2 + 2 * NH
        M, N = mc - 2 * NH, nc - 2 * NH
        mk2 = torch.zeros(mc, nc, dtype=torch.int8, device=mskp.device)
        mk2[NH:-NH, NH:-NH] = (_full_weight(mf, mc, nc) > 0.5).to(torch.int8)
        _fill(mk2)
        C = torch.zeros(9, mc, nc, dtype=torch.float64, device=mskp.device)

        def f(a, dj, di):
            return _odd(a, dj, di)[..., :M, :N]
        for l in range(9):
            w = 0.0
            for jj in (-1, 0, 1):
                for ii in (-1, 0, 1):
                    acc = 0.0
                    for kj in (-1, 0, 1):
                        for ki in (-1, 0, 1):
                            # coarse neighbour l's bilinear weight at the fine point
                            pj, pi = jj + kj - 2 * (l // 3 - 1), ii + ki - 2 * (l % 3 - 1)
                            if abs(pj) > 1 or abs(pi) > 1:
                                continue
                            acc = acc + (f(A[(ki + 1) + 3 * (kj + 1)], jj, ii)
                                         * f(mf, jj + kj, ii + ki)
                                         * (4 * cw[pj + 1] * cw[pi + 1]))
                    if torch.is_tensor(acc):
                        w = w + cw[jj + 1] * cw[ii + 1] * acc * f(mf, jj, ii)
            C[l, NH:-NH, NH:-NH] = w
        _at(C, NH, NH)[...] *= _at(mk2, NH, NH)
        A, mf, m, n = _fill(C), mk2.double(), mc, nc
        out.append((mk2, A))
    return out


def _offdiag(A, x, lo, hi):
    """Off-diagonal part of A x; the upper couplings by symmetry."""
    def p(k, dj=0, di=0):
        return _at(A[k], lo, hi, dj, di)

    def q(dj, di):
        return _at(x, lo, hi, dj, di)
    return (p(0) * q(-1, -1) + p(1) * q(-1, 0) + p(2) * q(-1, 1) + p(3) * q(0, -1)
            + p(3, 0, 1) * q(0, 1) + p(2, 1, -1) * q(1, -1) + p(1, 1, 0) * q(1, 0)
            + p(0, 1, 1) * q(1, 1))


def _smooth(msk, A, x, b):
    """Two damped-Jacobi sweeps (the first on the interior and one ring)."""
    for lo, hi in ((NH - 1, NH - 1), (NH, NH)):
        mk = _at(msk, lo, hi) != 0
        c3 = OMEGA / torch.where(mk, _at(A[4], lo, hi).abs(), 1.0)
        v = _at(x, lo, hi) * (1.0 - OMEGA) + c3 * (_offdiag(A, x, lo, hi) - _at(b, lo, hi))
        x = x.clone()
        _at(x, lo, hi)[...] = torch.where(mk, v, 0.0)
    return _fill(x)


def _residual(msk, A, x, b):
    r = torch.zeros_like(x)
    v = _at(b, NH, NH) - _offdiag(A, x, NH, NH) - _at(A[4], NH, NH) * _at(x, NH, NH)
    _at(r, NH, NH)[...] = torch.where(_at(msk, NH, NH) != 0, v, 0.0)
    return _fill(r)


def _restrict(msk2, r):
    c = torch.zeros(msk2.shape, dtype=torch.float64, device=r.device)
    c[NH:-NH, NH:-NH] = _full_weight(r, *msk2.shape) * (msk2[NH:-NH, NH:-NH] != 0)
    return _fill(c)


def _interp(msk1, msk2, x2):
    """Mask-weighted bilinear interpolation onto the fine array."""
    m2, n2 = x2.shape
    c2 = torch.tensor([0.0, 1.0, 0.5], dtype=torch.float64, device=x2.device)
    c3 = torch.tensor([0.0, 1.0, 0.5, float(np.float32(1.0) / np.float32(3.0)), 0.25],
                      dtype=torch.float64, device=x2.device)
    s = msk2.long()

    def q(a, dj, di):
        return a[1 + dj:m2 - 2 + dj, 1 + di:n2 - 2 + di]
    out = torch.zeros(msk1.shape, dtype=torch.float64, device=x2.device)
    for dj in (0, 1):
        for di in (0, 1):
            pts = [(0, 0)] + ([(0, 1)] if di else []) + ([(1, 0)] if dj else [])
            pts += [(1, 1)] if di and dj else []
            v = sum(q(x2, *p) for p in pts)
            if len(pts) > 1:
                v = v * (c2 if len(pts) == 2 else c3)[sum(q(s, *p) for p in pts)]
            out[dj:2 * (m2 - 3):2, di:2 * (n2 - 3):2] = v
    return out * (msk1 > 0)


def _vcycle(L, l, x, b):
    msk, A = L[l]
    if l == len(L) - 1:
        for _ in range(16):
            x = _smooth(msk, A, x, b)
        return x
    x = _smooth(msk, A, x, b)
    b2 = _restrict(L[l + 1][0], _residual(msk, A, x, b))
    x = x + _interp(msk, L[l + 1][0], _vcycle(L, l + 1, torch.zeros_like(b2), b2))
    return _smooth(msk, A, x, b)


def _fcycle(L, b):
    bs = [b]
    for mk, _ in L[1:]:
        bs.append(_restrict(mk, bs[-1]))
    x = _vcycle(L, len(L) - 1, torch.zeros_like(bs[-1]), bs[-1])
    for l in range(len(L) - 2, -1, -1):
        x = _vcycle(L, l, _interp(L[l][0], L[l + 1][0], x), bs[l])
    return x


def _norm(msk, x):
    return float((_at(x, NH, NH) * (_at(msk, NH, NH) != 0)).square().sum().sqrt())


def _solve(L, x, b, maxite=4, tol=1e-11):
    msk, A = L[0]
    r = _residual(msk, A, x, b)
    nb = _norm(msk, b)
    if not nb > 0:
        return x, 0.0
    res = _norm(msk, r) / nb
    for _ in range(maxite):
        if not res > tol:
            break
        x = x + _fcycle(L, r)
        r = _residual(msk, A, x, b)
        res = _norm(msk, r) / nb
    return x, res


def _w32(num, den):
    return float(np.float32(num) / np.float32(den))


def _edge(mk, q, vel, axis, cst, method, order):
    """Flux through the upper edges of the cells one below the interior to
    its last one, along `axis` of the interior's other extent."""
    m, n = q.shape

    def sh(a, k):
        if axis == 1:
            return a[NH:m - NH, NH - 1 + k:n - NH + k]
        return a[NH - 1 + k:m - NH + k, NH:n - NH]
    vel = sh(vel, 0)
    M = [sh(mk, k).long() for k in range(-2, 4)]
    Q = [sh(q, k) for k in range(-2, 4)]
    if order % 2 == 0:
        d, c = (-_w32(1, 12), _w32(7, 12)), (_w32(1, 60), -_w32(2, 15), _w32(37, 60))
        f = 0.5 * (Q[2] + Q[3])
        if order >= 4:
            f4 = d[0] * (Q[1] + Q[4]) + d[1] * (Q[2] + Q[3])
            if order == 4:
                f = torch.where(sum(M[1:5]) == 4, f4, f)
            else:
                f6 = c[0] * (Q[0] + Q[5]) + c[1] * (Q[1] + Q[4]) + c[2] * (Q[2] + Q[3])
                f = torch.where(sum(M) == 6, f6, f)
        f = vel * f
    else:
        UU = vel.abs()
        if method == 1:
            u1 = cst[4] * cst[3]
            if u1 > 0:
                UU = torch.where(UU < u1, vel * vel / (2.0 * u1) + 0.5 * u1, UU)
        d = (_w32(1, 30), -_w32(13, 60), _w32(47, 60), _w32(9, 20), -_w32(1, 20))
        c = (-_w32(1, 6), _w32(5, 6), _w32(2, 6))
        qp, qm = Q[2], Q[3]
        if order >= 3:
            qp = torch.where(sum(M[1:4]) == 3, c[0] * Q[1] + c[1] * Q[2] + c[2] * Q[3], qp)
            qm = torch.where(sum(M[2:5]) == 3, c[2] * Q[2] + c[1] * Q[3] + c[0] * Q[4], qm)
        if order == 5:
            qp = torch.where(sum(M[0:5]) == 5, sum(w * z for w, z in zip(d, Q[0:5])), qp)
            qm = torch.where(sum(M[1:6]) == 5, sum(w * z for w, z in zip(d[::-1], Q[1:6])), qm)
        f = 0.5 * (vel + UU) * qp + 0.5 * (vel - UU) * qm
    return torch.where(M[2] + M[3] == 2, f, 0.0)


def _advect(mk, q, u, v, cst, method, order, y):
    fx = _edge(mk, q, u, 1, cst, method, order)
    fy = _edge(mk, q, v, 0, cst, method, order)
    y[NH:-NH, NH:-NH] = -(fx[:, 1:] - fx[:, :-1]) / cst[0] - (fy[1:] - fy[:-1]) / cst[1]
    return _fill(y)


def _torque(mk, b, dx, gravity, dw):
    k = mk.long()
    c = _at(dw, NH, NH) * _at(k, NH, NH)
    on = (_at(k, NH, NH) + _at(k, NH, NH, 0, -1) == 2) & (_at(k, NH, NH, 0, 1) + _at(k, NH, NH) == 2)
    t = (_at(b, NH, NH, 0, 1) - _at(b, NH, NH, 0, -1)) * (0.5 * gravity / dx)
    _at(dw, NH, NH)[...] = c + torch.where(on, t, 0.0)
    return _fill(dw)


def _diffuse(mk, q, coef, dq):
    s = sum(_at(mk, NH, NH, *d) * (_at(q, NH, NH, *d) - _at(q, NH, NH))
            for d in ((0, -1), (0, 1), (-1, 0), (1, 0)))
    _at(dq, NH, NH)[...] += torch.where(_at(mk, NH, NH) == 1, coef * s, 0.0)
    return _fill(dq)


def _corner(x, out):
    out[:-1, :-1] = 0.25 * (x[:-1, :-1] + x[:-1, 1:] + x[1:, :-1] + x[1:, 1:])
    return out


def _ortho(mk, psi, dx, dy, u, v):
    k = mk.long()
    _at(u, 1, 1)[...] = torch.where(_at(k, 1, 1) + _at(k, 1, 1, 0, 1) == 2,
                                    (_at(psi, 1, 1, -1, 0) - _at(psi, 1, 1)) / dy, 0.0)
    _at(v, 1, 1)[...] = torch.where(_at(k, 1, 1) + _at(k, 1, 1, 1, 0) == 2,
                                    (_at(psi, 1, 1) - _at(psi, 1, 1, 0, -1)) / dx, 0.0)


class _Model:
    """One instance: state planes and the RK3_SSP step of the two models."""

    def __init__(self, p, g, fields, dev):
        self.p, self.g, self.euler = p, g, p.modelname == "euler"
        self.msk = torch.from_numpy(g.msk).to(dev)
        mskp = torch.zeros_like(self.msk)
        k = self.msk.long()
        mskp[:-1, :-1] = (k[:-1, :-1] + k[:-1, 1:] + k[1:, :-1] + k[1:, 1:] == 4).to(torch.int8)
        self.mskp = mskp
        self.L = _levels(mskp, g.dx, g.dy)
        nvar = 5 if self.euler else 6
        z = torch.zeros(nvar, g.nyl, g.nxl, dtype=torch.float64, device=dev)
        self.x, self.k = z, [z.clone() for _ in range(3)]
        self.x[0] = torch.from_numpy(fields["vorticity"])
        if not self.euler:
            self.x[4] = torch.from_numpy(fields["buoyancy"])
        self.work = torch.zeros_like(z[0])
        self.full()
        self.diagnose()

    def _finish(self, x, psi):
        x[1] = psi * self.mskp
        _ortho(self.msk, x[1], self.g.dx, self.g.dy, x[2], x[3])

    def full(self):
        psi, _ = _solve(self.L, self.x[1].clone(), _corner(self.x[0], self.work).clone())
        if self.g.geometry == "perio":
            psi = psi - _at(psi, NH, NH).mean()
        self._finish(self.x, psi)

    def fast(self, d):
        b = _corner(d[0], self.work).clone()
        psi = d[1].clone()
        for _ in range(2):
            psi = _vcycle(self.L, 0, psi, b)
        self._finish(d, psi)

    def diagnose(self):
        g = self.g
        u, v = self.x[2], self.x[3]
        on = _at(self.msk, NH, NH) == 1
        sp = ((_at(u, NH, NH) + _at(u, NH, NH, 0, -1)).abs()
              + (_at(v, NH, NH) + _at(v, NH, NH, -1, 0)).abs())
        ke = (_at(u, NH, NH) ** 2 + _at(u, NH, NH, 0, -1) ** 2 + _at(v, NH, NH) ** 2
              + _at(v, NH, NH, -1, 0) ** 2)
        self.umax = 0.5 * float(torch.where(on, sp, 0.0).max())
        self.ke = 0.25 * float(torch.where(on, ke, 0.0).sum()) / g.area
        self.ens = 0.5 * float(torch.where(on, _at(self.x[0], NH, NH) ** 2, 0.0).sum()) / g.area
        dtmax = _dtmax(g, self.p.modelname)
        self.dt = min(CFL * min(g.dx, g.dy) / self.umax, dtmax) if self.umax > 0 else dtmax

    def rhs(self, x, d, stage):
        p, g = self.p, self.g
        cst = [g.dx, g.dy, 0.05, self.umax, 0.0 if p.order % 2 == 0 else p.aparab]
        for q in (0,) if self.euler else (0, 4):
            _advect(self.msk, x[q], x[2], x[3], cst, 1, p.order, d[q])
        if self.euler:
            if stage != 2:
                self.fast(d)
            return
        _torque(self.msk, x[4], g.dx, p.gravity, d[0])
        if stage == 2 and p.diffusion:
            for q in (0, 4):
                _diffuse(self.msk, x[q], 1.5 * p.Kdiff / g.dx ** 2, d[q])
        self.fast(d)

    def step(self):
        k, x, dt = self.k, self.x, self.dt
        self.rhs(x, k[0], 0)
        self.rhs(x + dt * k[0], k[1], 1)
        self.rhs(x + 0.25 * dt * (k[0] + k[1]), k[2], 2)
        self.x = x + dt / 6.0 * (k[0] + k[1] + 4.0 * k[2])
        if self.euler:
            self.full()
        else:
            self.x[5] = self.x[4]
        self.diagnose()


def exact(case, seed):
    kind, dev = case["kind"], _dev()
    if kind in ("steps", "loop"):
        outs = []
        for p, g, f in _instances(case if kind == "steps" else dict(case, count=1), seed):
            o = _Model(p, g, f, dev)
            for _ in range(case["steps"]):
                o.step()
            outs.append(o)
        if kind == "steps":
            return [o.x for o in outs]
        o = outs[0]
        return {"state": o.x, "diags": [o.umax, o.ke, o.ens]}
    if kind in ("solve", "twov", "mg"):
        g, mskp, lev, x, b = _mg_inputs(case, seed, dev)
        if kind == "mg":
            (msk, A), (msk2, _) = lev
            x = _smooth(msk, A, x, b)
            r = _residual(msk, A, x, b)
            b2 = _restrict(msk2, r)
            x = _smooth(msk, A, x + _interp(msk, msk2, b2), b)
            return {"x": x, "r": r, "b2": b2}
        L = _levels(torch.from_numpy(mskp).to(dev), g.dx, g.dy)
        if kind == "twov":
            return {"x": _vcycle(L, 0, _vcycle(L, 0, x, b), b)}
        # the residual left after the last F-cycle is rounding and has no
        # value of its own
        return {"x": _solve(L, x, b)[0], "res": None}
    g, mk, w, b, psi, u, v, cst = _rhs_inputs(case, seed, dev)
    z = torch.zeros_like
    if kind == "rhs":
        dw, db, c, du, dv = z(w), z(w), z(w), z(w), z(w)
        for q, dq in ((w, dw), (b, db)):
            _advect(mk, q, u, v, cst, 1, case["order"], dq)
        _torque(mk, b, g.dx, 1.0, dw)
        for q, dq in ((w, dw), (b, db)):
            _diffuse(mk, q, 1e-5 / g.dx ** 2, dq)
        _corner(dw, c)
        _ortho(mk, psi, g.dx, g.dy, du, dv)
        return [dw, db, c, du, dv]
    on = (_at(mk, NH, NH) == 1).double()
    s = (_at(u, NH, NH), _at(u, NH, NH, 0, -1), _at(v, NH, NH), _at(v, NH, NH, -1, 0))
    W, Bq = _at(w, NH, NH), _at(b, NH, NH)
    ke = 0.25 * float((on * sum(a * a for a in s)).sum())
    maxu = 0.5 * float((on * ((s[0] + s[1]).abs() + (s[2] + s[3]).abs())).max())
    z1, z2 = float((on * W).sum()), float((on * W * W).sum())
    return [ke, maxu, z1, z2, z2, float((on * W * Bq).sum()), float((on * Bq).sum()),
            float(_at(psi, NH, NH).sum())]
