"""The work that programs built on this package have it do, as cases to time.

A case is a dict of plain values; ``prepare`` builds what a program holds
before a call (containers, velocity, fields, plans), ``run`` is one pass
through the public entry points, ``work`` the bytes and operations a pass
cannot do without, ``exact`` the values of a pass in plain 64-bit torch where
a closed computation gives them.

Kinds of case:

* ``step``: one time step of a particle-in-cell program: ``advection!``,
  ``move_particles!``, ``inject_particles!`` (where the program injects) and
  ``particle2grid!``;
* ``phases``: one step of a multi-material program: advection, move, the phase
  injection and ``update_phase_ratios!``;
* ``schemes``: one step of a program that carries particles with the MQS or
  LinP velocity interpolation and a nodal field by semi-Lagrangian advection;
* ``transfers``: the transfers between grid and particles around an implicit
  solve: ``grid2particle!``, ``grid2particle_flip!``, the centroid transfers
  and ``particle2grid!`` of several fields;
* ``adjoint``: one gradient of an inverse problem (forward and pullback);
* ``ensemble``: one captured step of a batch of independent 2D grids.

States in a time loop start a few steps in, so that cells are uneven, slots
have holes and the injection has cells to fill.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "justpic.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import justpic_hip as jp  # noqa: E402
from justpic_hip.configs import gaussian_T, inverse2d, sample, vertex_axes  # noqa: E402

SPIN_UP = 8  # steps a time loop has taken before the first timed one


def listed():
    return [
        # The smallest useful grid, with the package's default synchronous
        # calls: a test or a teaching script, bound by launches and waits.
        dict(name="step2d_f64_32_sync", kind="step", form="f64", axes="readme", nx=32, ny=32, nz=0,
             nxcell=24, max_xcell=48, min_xcell=12, method="rk2", alpha=0.5, cfl=1.0, fields=1,
             inject=True, sync=True),
        # The rotating cell of the README at its own size and on its own
        # rounded axes, in the FP32-split form.
        dict(name="step2d_split_256_readme", kind="step", form="split", axes="readme", nx=256,
             ny=256, nz=0, nxcell=24, max_xcell=48, min_xcell=12, method="rk2", alpha=0.5, cfl=1.0,
             fields=1, inject=True, sync=False),
        # The temperature advection that bench.py times by default.
        dict(name="step2d_split_512", kind="step", form="split", axes="lin", nx=512, ny=512, nz=0,
             nxcell=24, max_xcell=48, min_xcell=12, method="rk2", alpha=0.5, cfl=1.0, fields=1,
             inject=True, sync=False),
        # The same in FP64, what a caller of the reference gets by switching.
        dict(name="step2d_f64_512", kind="step", form="f64", axes="lin", nx=512, ny=512, nz=0,
             nxcell=24, max_xcell=48, min_xcell=12, method="rk2", alpha=0.5, cfl=1.0, fields=1,
             inject=True, sync=False),
        # A refined grid (vector axes) of odd size with RK4 and three fields
        # on the particles, as a thermo-chemical model has them.
        dict(name="step2d_f64_refined_389x211", kind="step", form="f64", axes="vector", nx=389,
             ny=211, nz=0, nxcell=24, max_xcell=48, min_xcell=12, method="rk4", alpha=0.5, cfl=0.8,
             fields=3, inject=True, sync=False),
        # The largest: 128^3 cells, 65 M particles, in the FP32-split form.
        dict(name="step3d_split_128", kind="step", form="split", axes="lin", nx=128, ny=128, nz=128,
             nxcell=27, max_xcell=54, min_xcell=14, method="rk2", alpha=0.5, cfl=1.0, fields=1,
             inject=False, sync=False),
        # An ordinary 3D model of ragged size in FP64: RK4, two fields,
        # injection.
        dict(name="step3d_f64_61x47x74", kind="step", form="f64", axes="lin", nx=61, ny=47, nz=74,
             nxcell=27, max_xcell=54, min_xcell=14, method="rk4", alpha=0.5, cfl=0.8, fields=2,
             inject=True, sync=False),
        # A multi-material 2D model: three phases and a temperature.
        dict(name="phases2d_384x257", kind="phases", axes="lin", nx=384, ny=257, nz=0, nxcell=24,
             max_xcell=48, min_xcell=12, method="rk2", alpha=0.5, cfl=0.8, fields=1, phases=3,
             sync=False),
        # Composition on particles with MQS velocities, temperature carried on
        # the nodes by backtracking.
        dict(name="schemes2d_mqs_300x431", kind="schemes", axes="lin", scheme="mqs", nx=300, ny=431,
             nz=0, nxcell=24, max_xcell=48, min_xcell=12, method="rk2", alpha=0.5, cfl=0.5, fields=1,
             sync=False),
        # Grid-particle transfers of a model with a FLIP temperature, a centred
        # and two nodal fields.
        dict(name="transfers2d_f64_512x384", kind="transfers", form="f64", axes="lin", nx=512,
             ny=384, nz=0, nxcell=24, max_xcell=48, min_xcell=12, fields=2, sync=False),
        # The velocity inversion of bench.py --case adjoint: 1 M particles, 100
        # RK2 steps, checkpoints every 10.
        dict(name="adjoint2d_256", kind="adjoint", form="f64", nx=256, nxcell=16, max_xcell=32,
             min_xcell=8, method="rk2", steps=100, every=10, sync=False),
        # A parameter study: 12 independent grids of uneven size, one graph
        # launch per step.
        dict(name="ensemble_12", kind="ensemble", members=12, smallest=64, largest=512, nxcell=24,
             max_xcell=48, min_xcell=12, cfl=1.0, sync=False),
    ]


# (nxcell, max_xcell, min_xcell) that the tests and workloads use
_FILLS = {2: ((24, 48, 12), (24, 48, 12), (12, 24, 5), (16, 32, 8), (32, 64, 16)),
          3: ((27, 54, 14), (27, 54, 14), (24, 48, 12), (16, 32, 8))}


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def _shape(rng, D, lo, hi):
    """D uneven cell counts whose product lies between lo and hi."""
    cells = _log(rng, lo, hi)
    f = [rng.uniform(0.75, 1.33) for _ in range(D)]
    s = (cells / math.prod(f)) ** (1.0 / D)
    n = [max(8, int(s * x)) for x in f]
    return n + [0] * (3 - D)


def draw(rng):
    kind = rng.choice(("step", "step", "step", "step", "phases", "schemes", "transfers", "adjoint",
                       "ensemble"))
    cfl = round(rng.uniform(0.5, 1.0), 2)
    if kind == "ensemble":
        lo = rng.choice((48, 64, 96))
        return dict(kind=kind, members=rng.randint(4, 12), smallest=lo,
                    largest=rng.choice((192, 256, 384, 512)), nxcell=24, max_xcell=48, min_xcell=12,
                    cfl=cfl, sync=False)
    if kind == "adjoint":
        method = rng.choice(("rk2", "rk2", "rk4"))
        return dict(kind=kind, form=rng.choice(("f64", "split")), nx=int(_log(rng, 24, 256)),
                    nxcell=16, max_xcell=32, min_xcell=8, method=method,
                    steps=rng.randint(8, 80 if method == "rk2" else 40),
                    every=rng.choice((4, 10, 16)), sync=False)
    D = rng.choice((2, 2, 3))
    nxcell, K, mn = rng.choice(_FILLS[D])
    axes = rng.choice(("lin", "lin", "readme", "vector"))
    form = rng.choice(("f64", "split"))
    method = rng.choice(("rk2", "rk2", "rk4", "euler"))
    common = dict(nxcell=nxcell, max_xcell=K, min_xcell=mn)
    if kind in ("phases", "schemes") or axes == "vector":
        form = "f64"
    hi = {2: 512 * 512, 3: 96 ** 3 if form == "split" else 72 ** 3}[D]
    if kind in ("phases", "schemes"):
        hi = {2: 420 * 420, 3: 40 ** 3}[D]
    nx, ny, nz = _shape(rng, D, {2: 24 * 24, 3: 10 ** 3}[D], hi)
    common.update(axes=axes, nx=nx, ny=ny, nz=nz, sync=rng.random() < 0.15)
    step = dict(method=method, alpha=rng.choice((0.5, 0.5, 2.0 / 3.0)), cfl=cfl,
                fields=rng.randint(1, 3))
    if kind == "step":
        return dict(kind=kind, form=form, inject=rng.random() < 0.75, **common, **step)
    if kind == "phases":
        return dict(kind=kind, phases=rng.randint(2, 6), **common, **step)
    if kind == "schemes":
        step["method"] = rng.choice(("rk2", "rk4"))
        step["cfl"] = 0.5 * cfl
        return dict(kind=kind, scheme=rng.choice(("mqs", "linp", "linear")), **common, **step)
    return dict(kind=kind, form=form, fields=rng.randint(1, 3), **common)


# ---------------------------------------------------------------- building

_contexts = {}


def _context(case):
    """One context per process and launch mode, as a program has it."""
    sync = bool(case["sync"])
    if sync not in _contexts:
        _contexts[sync] = jp.Context(0, synchronous=sync)
    return _contexts[sync]


class _Span:
    def __init__(self, owner, shape, strides=None):
        self.owner = owner
        d = owner if isinstance(owner, jp.DeviceArray) else owner.data
        self.__cuda_array_interface__ = {
            "shape": shape, "strides": strides, "typestr": d.dtype.str,
            "data": (d.ptr, False), "version": 3}


def _view(a):
    """A torch tensor over the device buffer of a DeviceArray (Julia order:
    first dimension contiguous) or a CellArray (slot, cell)."""
    if isinstance(a, jp.DeviceArray):
        return torch.as_tensor(_Span(a, tuple(reversed(a.shape))), device="cuda")
    return torch.as_tensor(_Span(a, (a.K, a.C)), device="cuda")


def _dims(case):
    return (case["nx"], case["ny"], case["nz"]) if case["nz"] else (case["nx"], case["ny"])


def _axes(case):
    n = _dims(case)
    if case["axes"] == "vector":  # refined towards the middle by up to 1.7 to 1
        xi = [np.linspace(0.0, 1.0, m + 1) for m in n]
        return tuple(jp.Axis(x + 0.25 * np.sin(2 * np.pi * x) / (2 * np.pi), "vector") for x in xi)
    return vertex_axes(n, readme=case["axes"] == "readme")


def _flow(xi_vel, rng):
    """The stream-function cell (2D) or the cellular flow (3D) at a seeded
    amplitude, with a seeded smooth variation that keeps the walls closed."""
    amp, e, pi = float(rng.uniform(200.0, 250.0)), float(rng.uniform(-0.1, 0.1)), np.pi
    s, c = np.sin, np.cos
    if len(xi_vel) == 2:
        f = (lambda x, y: amp * (s(pi * x) * c(pi * y) + 2 * e * s(2 * pi * x) * c(2 * pi * y)),
             lambda x, y: -amp * (c(pi * x) * s(pi * y) + 2 * e * c(2 * pi * x) * s(2 * pi * y)))
    else:
        f = (lambda x, y, z: amp * s(pi * x) * c(pi * y) * c(pi * z) * (1 + e),
             lambda x, y, z: amp * c(pi * x) * s(pi * y) * c(pi * z) * (1 - e),
             lambda x, y, z: -2 * amp * c(pi * x) * c(pi * y) * s(pi * z))
    return tuple(sample(g, a) for g, a in zip(f, xi_vel))


def _time_step(xv, V, cfl):
    return cfl * min(float(np.min(a.dx)) / float(np.abs(v).max()) for a, v in zip(xv, V))


def _integrator(case):
    return {"euler": jp.Euler, "rk2": lambda: jp.RungeKutta2(case.get("alpha", 0.5)),
            "rk4": jp.RungeKutta4}[case["method"]]()


def _nodal_values(xv, rng, f):
    """A smooth nodal field: a Gaussian at a seeded place plus a wave."""
    x0, y0 = rng.uniform(0.3, 0.7, 2)
    if len(xv) == 2:
        return gaussian_T(xv, x0, y0, 0.02 + 0.02 * f) + 0.1
    k = float(rng.uniform(2.0, 5.0))
    return sample(lambda x, y, z: np.exp(-((x - x0) ** 2 + (y - y0) ** 2) / 0.05) *
                  (1.0 + 0.3 * np.sin(k * z + f)) + 0.1, xv)


class _State:
    pass


def _container(case, seed):
    """Particles, velocity, time step and fields of a program before its loop."""
    s = _State()
    rng = np.random.default_rng(seed)
    s.case, s.rng, s.ctx = case, rng, _context(case)
    s.xv = _axes(case)
    s.xi = jp.staggered_grid(s.xv, readme=case["axes"] == "readme")
    s.p = jp.init_particles(s.ctx, case["nxcell"], case["max_xcell"], case["min_xcell"], *s.xi,
                            seed=int(seed), form=case.get("form", "f64"))
    V = _flow(s.xi, rng)
    s.dt = _time_step(s.xv, V, case.get("cfl", 0.8))
    s.V = tuple(jp.DeviceArray.from_host(s.ctx, v) for v in V)
    s.T = [jp.DeviceArray.from_host(s.ctx, _nodal_values(s.xv, rng, f))
           for f in range(case["fields"])]
    s.Fp = [jp.CellArray(s.ctx, s.p.ni, s.p.max_xcell, fill=float("nan")) for _ in s.T]
    for fp, t in zip(s.Fp, s.T):
        jp.grid2particle_(fp, t, s.p)
    return s


def _step(s):
    p, fields = s.p, tuple(s.Fp)
    jp.advection_(p, s.rk, s.V, s.dt)
    jp.move_particles_(p, fields)
    if s.case.get("inject", True):
        jp.inject_particles_(p, fields)


def _to_grid(s):
    if len(s.T) == 1:
        jp.particle2grid_(s.T[0], s.Fp[0], s.p)
    else:
        jp.particle2grid_(tuple(s.T), tuple(s.Fp), s.p)


def _views(s, *more):
    s.out = {"coords": [_view(c) for c in s.p.coords], "index": _view(s.p.index),
             "fields": [_view(f) for f in s.Fp], "nodal": [_view(t) for t in s.T]}
    for name, arrays in more:
        s.out[name] = [_view(a) for a in arrays]


def _prepare_step(case, seed):
    s = _container(case, seed)
    s.rk = _integrator(case)
    for _ in range(SPIN_UP):
        _step(s)
        _to_grid(s)
    _views(s)
    return s


def _prepare_phases(case, seed):
    s = _container(case, seed)
    s.rk = _integrator(case)
    p, n = s.p, case["phases"]
    s.phases = jp.CellArray(s.ctx, p.ni, p.max_xcell, fill=float("nan"))
    s.ratios = jp.PhaseRatios(s.ctx, n, p.ni)
    s.ctx.sync()
    # layers with a wavy boundary: the phase of each particle by its place
    x, y = _view(p.coords[0]), _view(p.coords[-1])
    layer = (n * (y + 0.06 * torch.sin(2 * math.pi * x + float(s.rng.uniform(0, 6))))).floor()
    _view(s.phases).copy_(layer.clamp(0, n - 1) + 1)
    torch.cuda.synchronize()
    for _ in range(SPIN_UP):
        _phase_step(s)
    _views(s, ("phases", [s.phases]), ("ratios", [s.ratios.fields[k] for k in s.ratios.fields]))
    return s


def _phase_step(s):
    p = s.p
    jp.advection_(p, s.rk, s.V, s.dt)
    jp.move_particles_(p, (s.phases,) + tuple(s.Fp))
    jp.inject_particles_phase_(p, s.phases, tuple(s.Fp), tuple(s.T))
    jp.update_phase_ratios_(s.ratios, p, s.phases)


def _prepare_schemes(case, seed):
    s = _container(case, seed)
    s.rk = _integrator(case)
    s.back = jp.BacktrackGrid(s.ctx, s.xi, s.xv)
    s.T0 = [t.copy() for t in s.T]
    scheme = case["scheme"]
    s.advect = {"linear": jp.advection_, "mqs": jp.advection_MQS_,
                "linp": jp.advection_LinP_}[scheme]
    s.backtrack = {"linear": jp.semilagrangian_advection_,
                   "mqs": jp.semilagrangian_advection_MQS_,
                   "linp": jp.semilagrangian_advection_LinP_}[scheme]
    for _ in range(SPIN_UP):
        _scheme_step(s)
    _views(s)
    return s


def _scheme_step(s):
    s.advect(s.p, s.rk, s.V, s.dt)
    jp.move_particles_(s.p, tuple(s.Fp))
    jp.inject_particles_(s.p, tuple(s.Fp))
    if len(s.T) == 1:
        s.backtrack(s.T[0], s.T0[0], s.rk, s.V, s.xi, s.back, s.dt)
    else:
        s.backtrack(tuple(s.T), tuple(s.T0), s.rk, s.V, s.xi, s.back, s.dt)


def _prepare_transfers(case, seed):
    s = _container(case, seed)
    s.rk = jp.RungeKutta2()
    for _ in range(3):
        _step(s)
    p = s.p
    s.T0 = [t.copy() for t in s.T]  # before and after the solve
    s.F = [jp.DeviceArray.from_host(s.ctx, _nodal_values(s.xv, s.rng, f)) for f in range(len(s.T))]
    s.Gp = [jp.CellArray(s.ctx, p.ni, p.max_xcell, fill=float("nan")) for _ in s.T]
    if p.form == "f64":
        s.Hp = [jp.CellArray(s.ctx, p.ni, p.max_xcell, fill=float("nan")) for _ in s.T]
        for hp, t in zip(s.Hp, s.T):
            jp.grid2particle_(hp, t, p)
        xc = [a.x for a in p.xci]
        mesh = np.meshgrid(*xc, indexing="ij")
        k = float(s.rng.uniform(3.0, 6.0))
        s.Fc = jp.centroid_field(p, np.sin(k * mesh[0]) * np.cos(4 * mesh[-1]))
        s.Cp = jp.CellArray(s.ctx, p.ni, p.max_xcell, fill=float("nan"))
        s.Gc = jp.centroid_field(p)
    s.ctx.sync()
    s.out = {"g2p": [_view(a) for a in s.Gp], "p2g": [_view(t) for t in s.T]}
    if p.form == "f64":
        s.out.update(flip=[_view(a) for a in s.Hp], c2p=_view(s.Cp), p2c=_view(s.Gc))
    return s


def _transfers(s):
    p = s.p
    jp.grid2particle_(tuple(s.Gp), tuple(s.F), p)
    if p.form == "f64":
        jp.grid2particle_flip_(tuple(s.Hp), tuple(s.F), tuple(s.T0), p, alpha=0.1)
        jp.centroid2particle_(s.Cp, s.Fc, p)
        jp.particle2centroid_(s.Gc, s.Fp[0], p)
    _to_grid(s)


def _prepare_adjoint(case, seed):
    s = _State()
    s.case, s.ctx = case, _context(case)
    cfg = inverse2d(case["nx"], seed=int(seed) % (1 << 31))
    p = jp.init_particles(s.ctx, case["nxcell"], case["max_xcell"], case["min_xcell"],
                          *cfg["xi_vel"], seed=int(seed))
    s.p, s.xv, s.xi = p, cfg["xv"], cfg["xi_vel"]
    s.x0, s.Tp = jp.flatten(p)
    x, y = (a.to_host() for a in s.x0)
    s.Tp.copy_from(cfg["T"](x, y))
    s.dt = cfg["dt"]
    s.V = tuple(jp.DeviceArray.from_host(s.ctx, v) for v in cfg["V"])
    Vt = tuple(jp.DeviceArray.from_host(s.ctx, v) for v in cfg["V_true"])
    s.op = jp.AdvectionP2G(p, _integrator(case), s.dt, case["steps"], case["every"],
                           form=case["form"])
    target = s.op.forward(Vt, s.x0, s.Tp).flat()
    _, fb = jp.l2_loss(s.op.forward(s.V, s.x0, s.Tp), target)
    s.Fbar = jp.DeviceArray.from_host(s.ctx, fb.reshape(s.op.nodes, order="F"))
    s.grads = s.op.pullback(s.Fbar)
    F = s.op.forward(s.V, s.x0, s.Tp)
    Vbar, xbar, Tbar = s.grads
    s.ctx.sync()
    s.out = {"F": _view(F), "Vbar": [_view(v) for v in Vbar], "x0bar": [_view(v) for v in xbar],
             "Tpbar": _view(Tbar)}
    return s


def _sizes(case):
    """Cell counts per side of the members: spread over the range, uneven."""
    m, a, b = case["members"], case["smallest"], case["largest"]
    return [int(round(a * (b / a) ** ((i * 5 % m) / max(1, m - 1)))) for i in range(m)]


class _Members(_State):
    graph = None

    def __del__(self):
        if self.graph is not None:
            self.ctx.sync()
            self.ctx.graph_destroy(self.graph)
            self.ens.close()


def _prepare_ensemble(case, seed):
    s = _Members()
    rng = np.random.default_rng(seed)
    s.case, s.ctx = case, _context(case)
    members, s.fields, s.nodal = [], [], []
    for i, n in enumerate(_sizes(case)):
        xv = vertex_axes((n, n))
        xi = jp.staggered_grid(xv)
        p = jp.init_particles(s.ctx, case["nxcell"], case["max_xcell"], case["min_xcell"], *xi,
                              seed=int(seed) * 100 + i, form="split")
        V = _flow(xi, rng)
        T = jp.DeviceArray.from_host(s.ctx, _nodal_values(xv, rng, 0))
        f = jp.CellArray(s.ctx, p.ni, p.max_xcell, fill=float("nan"))
        jp.grid2particle_(f, T, p)
        members.append((p, tuple(jp.DeviceArray.from_host(s.ctx, v) for v in V),
                        _time_step(xv, V, case["cfl"])))
        s.fields.append(f)
        s.nodal.append(T)
    s.ens = jp.Ensemble(s.ctx, members)
    s.ens.step(s.fields, s.nodal)
    s.ctx.sync()
    s.graph = s.ens.capture_step(s.fields, s.nodal)
    for _ in range(SPIN_UP):
        s.ctx.graph_launch(s.graph)
    s.ctx.sync()
    s.out = [{"offsets": [_view(c) for c in p.coords], "index": _view(p.index), "field": _view(f),
              "nodal": _view(T)} for (p, _, _), f, T in zip(members, s.fields, s.nodal)]
    return s


def prepare(case, seed):
    s = {"step": _prepare_step, "phases": _prepare_phases, "schemes": _prepare_schemes,
         "transfers": _prepare_transfers, "adjoint": _prepare_adjoint,
         "ensemble": _prepare_ensemble}[case["kind"]](case, seed)
    s.ctx.sync()
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "step":
        _step(s)
        _to_grid(s)
    elif kind == "phases":
        _phase_step(s)
    elif kind == "schemes":
        _scheme_step(s)
    elif kind == "transfers":
        _transfers(s)
    elif kind == "adjoint":
        s.op.forward(s.V, s.x0, s.Tp)
        s.op.pullback(s.Fbar, s.grads)
    else:
        s.ctx.graph_launch(s.graph)
    return s.out


# ---------------------------------------------------------------- work

def work(case):
    """Every input read once and every output written once; operations of the
    interpolations (2^D - 1 lerps of 2 operations) and of the nodal weights."""
    stages = {"euler": 1, "rk2": 2, "rk4": 4}.get(case.get("method", "rk2"))
    kind = case["kind"]
    if kind == "ensemble":
        b = f = 0
        for n in _sizes(case):
            w = work(dict(kind="step", form="split", nx=n, ny=n, nz=0, nxcell=case["nxcell"],
                          max_xcell=case["max_xcell"], method="rk2", fields=1))
            b, f = b + w["bytes"], f + w["flops"]
        return {"bytes": b, "flops": f}
    if kind == "adjoint":
        n = case["nx"]
        P, Vn, Nn, N = n * n * case["nxcell"], 2 * (n + 1) * (n + 2), (n + 1) ** 2, case["steps"]
        # inputs x0, Tp, V, Fbar; outputs F, Vbar, x0bar, Tpbar
        return {"bytes": 8 * (P * (2 + 1) + Vn + Nn) + 8 * (Nn + Vn + P * (2 + 1)),
                "flops": P * N * stages * 2 * (3 * 3 + 4) * 3}
    n = _dims(case)
    D, C = len(n), math.prod(n)
    nq = 2 ** D
    nxcell = -(-case["nxcell"] // nq) * nq
    S, P = C * max(nxcell, case["max_xcell"]), C * nxcell
    w = 4 if case.get("form") == "split" else 8
    nF = case["fields"]
    Nn = math.prod(m + 1 for m in n)
    Vb = 8 * sum(math.prod(m + (1 if d == c else 2) for d, m in enumerate(n)) for c in range(D))
    lerp = 3 * (nq - 1) + 2 * D
    weights = P * nq * (3 * D + 2 + 2 * nF)
    if kind == "transfers":
        b = S + P * D * w + 2 * nF * 8 * Nn + P * nF * 16
        f = P * nF * lerp + weights
        if case["form"] == "f64":
            b += P * nF * 16 + 8 * nF * Nn + P * 8 + 2 * 8 * C
            f += P * (2 * nF * lerp + lerp + 3 * D + 2)
        return {"bytes": b, "flops": f}
    b = 2 * S + 2 * P * (D * w + 8 * nF) + Vb
    f = P * stages * D * (lerp + 2)
    if kind == "step":
        return {"bytes": b + 8 * nF * Nn, "flops": f + weights}
    if kind == "schemes":
        return {"bytes": b + 16 * nF * Nn, "flops": 2 * f + Nn * (stages * D * lerp + nF * lerp)}
    L = C + Nn + sum(math.prod(m + (1 if d == c else 0) for d, m in enumerate(n)) for c in range(D))
    if D == 3:
        L += sum(math.prod(m + (0 if d == c else 1) for d, m in enumerate(n)) for c in range(D))
    return {"bytes": b + 16 * P + 8 * nF * Nn + 8 * case["phases"] * L,
            "flops": f + P * (2 ** D + D + 1) * 3 * D}


# ---------------------------------------------------------------- exact values

def _bracket(x, p):
    return (torch.searchsorted(x, p.contiguous(), right=True) - 1).clamp(0, x.numel() - 2)


def _lerp(F, idx, t):
    """Multilinear interpolation of F (reversed dims: last index fastest) at
    the cells idx (one index per dimension, first dimension first)."""
    D = len(idx)
    out = 0.0
    for q in range(1 << D):
        w, at = 1.0, []
        for d in range(D):
            b = (q >> d) & 1
            w = w * (t[d] if b else 1.0 - t[d])
            at.append(idx[d] + b)
        out = out + w * F[tuple(reversed(at))]
    return out


def _axis(a):
    return torch.from_numpy(np.array(a.x)).cuda(), torch.from_numpy(np.array(a.dx)).cuda()


def _positions(s):
    """(positions, cells, t, active mask) of a container's slots, 64 bits."""
    p, D = s.p, s.p.D
    n = p.ni
    act = _view(p.index) != 0
    c = torch.arange(p.C, device="cuda")
    cell = []
    for m in n:
        cell.append(c % m)
        c = c // m
    pos, t, idx = [], [], []
    for d in range(D):
        x, dx = _axis(s.xv[d])
        i = cell[d].expand(p.max_xcell, -1)
        u = _view(p.coords[d]).double()
        if p.form == "split":
            pos.append(x[i] + u * dx[i])
            t.append(u)
        else:
            pos.append(u)
            t.append((u - x[i]) / dx[i])
        idx.append(i)
    return pos, idx, t, act


def _gather_nodes(nodes, pos, cell, values, xs, rel=None):
    """Sums over particles of 1/|x - x_node|^2 and of that times each value, at
    the 2^D nodes around each particle's cell."""
    D = len(pos)
    W = torch.zeros(math.prod(nodes), dtype=torch.float64, device="cuda")
    S = [torch.zeros_like(W) for _ in values]
    for q in range(1 << D):
        lin, stride, d2 = 0, 1, 0.0
        for d in range(D):
            b = (q >> d) & 1
            i = cell[d] + b
            lin = lin + i * stride
            stride *= nodes[d]
            dist = pos[d] - xs[d][i] if rel is None else (rel[d][0] - b) * rel[d][1]
            d2 = d2 + dist * dist
        w = 1.0 / d2
        W.index_add_(0, lin, w)
        for acc, v in zip(S, values):
            acc.index_add_(0, lin, w * v)
    return W, S


def _exact_transfers(case, seed):
    s = prepare(case, seed)
    p, D = s.p, s.p.D
    pos, idx, t, act = _positions(s)
    nan = float("nan")
    F = [_view(f) for f in s.F]
    out = {"g2p": [torch.where(act, _lerp(f, idx, t), nan) for f in F]}
    sel = [x[act] for x in pos]
    cell = [i[act] for i in idx]
    vals = [_view(f)[act] for f in s.Fp]
    xs = [_axis(a)[0] for a in s.xv]
    nodes = tuple(m + 1 for m in p.ni)
    rel = None
    if p.form == "split":  # distances from the offsets, free of cancellation
        rel = [(u[act], _axis(a)[1][i]) for u, a, i in zip(t, s.xv, cell)]
    W, S = _gather_nodes(nodes, sel, cell, vals, xs, rel)
    out["p2g"] = [(v / W).reshape(tuple(reversed(nodes))) for v in S]
    if p.form == "f64":
        al = 0.1
        flip = []
        for hp, f, t0 in zip(s.Hp, F, s.T0):
            new, old = _lerp(f, idx, t), _lerp(_view(t0), idx, t)
            flip.append(torch.where(act, new * al + (_view(hp) + new - old) * (1.0 - al), nan))
        out["flip"] = flip
        xc = [_axis(a) for a in p.xci]
        ci, ct = [], []
        for d in range(D):
            x, dx = xc[d]
            k = torch.where(pos[d] < x[idx[d]], idx[d] - 1, idx[d]).clamp(0, p.ni[d] - 2)
            ci.append(k)
            ct.append((pos[d] - x[k]) / dx[k])
        out["c2p"] = torch.where(act, _lerp(_view(s.Fc), ci, ct), nan)
        w = 1.0
        for d in range(D):
            dx = _axis(s.xv[d])[1]
            w = w * (1.0 - (pos[d] - xc[d][0][idx[d]]).abs() / dx[idx[d]])
        w = torch.where(act, w, 0.0)
        v = torch.where(act, _view(s.Fp[0]), 0.0)
        out["p2c"] = ((w * v).sum(0) / w.sum(0)).reshape(tuple(reversed(p.ni)))
    return out


def _velocity(grid, V, x):
    out = []
    for axes, v in zip(grid, V):
        idx, t = [], []
        for (ax, dx), xd in zip(axes, x):
            k = _bracket(ax, xd.detach())
            idx.append(k)
            t.append((xd - ax[k]) / dx[k])
        out.append(_lerp(v, idx, t))
    return out


def _trajectory(method, steps, dt, grid, V, x, lo, hi):
    alive = torch.ones_like(x[0], dtype=torch.bool)
    for _ in range(steps):
        k1 = _velocity(grid, V, x)
        if method == "rk2":
            k2 = _velocity(grid, V, [a + 0.5 * dt * k for a, k in zip(x, k1)])
            new = [a + dt * k for a, k in zip(x, k2)]
        elif method == "rk4":
            k2 = _velocity(grid, V, [a + 0.5 * dt * k for a, k in zip(x, k1)])
            k3 = _velocity(grid, V, [a + 0.5 * dt * k for a, k in zip(x, k2)])
            k4 = _velocity(grid, V, [a + dt * k for a, k in zip(x, k3)])
            new = [a + dt * (p + 2 * q + 2 * r + u) / 6
                   for a, p, q, r, u in zip(x, k1, k2, k3, k4)]
        else:
            new = [a + dt * k for a, k in zip(x, k1)]
        for d in range(len(x)):
            n = new[d].detach()
            alive = alive & (n > lo[d]) & (n < hi[d])
        x = [torch.where(alive, n, a) for n, a in zip(new, x)]
    return x, alive


def _exact_adjoint(case, seed):
    if case["form"] != "f64":  # float32 trajectories: 64 bits follow another path
        return None
    s = prepare(case, seed)
    xs = [_axis(a)[0] for a in s.xv]
    lo, hi = [float(x[0]) for x in xs], [float(x[-1]) for x in xs]
    grid = [[_axis(a) for a in g] for g in s.xi]
    V = [_view(v).clone() for v in s.V]
    x0, Tp, Fbar = [_view(a) for a in s.x0], _view(s.Tp), _view(s.Fbar).reshape(-1)
    nodes, method, steps = s.op.nodes, case["method"], case["steps"]
    chunk = 1 << 18
    ends, W, S = [], 0.0, 0.0
    with torch.no_grad():
        for a in range(0, Tp.numel(), chunk):
            x, alive = _trajectory(method, steps, s.dt, grid, V, [v[a:a + chunk] for v in x0],
                                   lo, hi)
            x, T = [v[alive] for v in x], Tp[a:a + chunk][alive]
            w, (v,) = _gather_nodes(nodes, x, [_bracket(g, u) for g, u in zip(xs, x)], [T], xs)
            W, S = W + w, S + v
            ends.append(alive)
        F = S / W
        scale = torch.where(W > 0, Fbar / W, 0.0)
        Ff = torch.where(W > 0, F, 0.0)
    Vg = [v.requires_grad_(True) for v in V]
    xbar, Tbar = [[] for _ in x0], []
    for n, a in enumerate(range(0, Tp.numel(), chunk)):
        start = [v[a:a + chunk].clone().requires_grad_(True) for v in x0]
        T = Tp[a:a + chunk].clone().requires_grad_(True)
        x, _ = _trajectory(method, steps, s.dt, grid, Vg, start, lo, hi)
        alive = ends[n]
        x, Ta = [v[alive] for v in x], T[alive]
        # dF = sum over particles of (T - F) dw / W + w dT / W
        total = 0.0
        cell = [_bracket(g, u.detach()) for g, u in zip(xs, x)]
        for q in range(4):
            i, j = cell[0] + (q & 1), cell[1] + (q >> 1)
            lin = i + nodes[0] * j
            w = 1.0 / ((x[0] - xs[0][i]) ** 2 + (x[1] - xs[1][j]) ** 2)
            total = total + (w * (Ta - Ff[lin]) * scale[lin]).sum()
        total.backward()
        for d, v in enumerate(start):
            xbar[d].append(v.grad)
        Tbar.append(T.grad)
    return {"F": F.reshape(tuple(reversed(nodes))), "Vbar": [v.grad for v in Vg],
            "x0bar": [torch.cat(v) for v in xbar], "Tpbar": torch.cat(Tbar)}


def exact(case, seed):
    """In 64 bits with torch: the transfers and the gradient.  A time step has
    no such value: slots, drops and injected copies follow sequential rules."""
    if case["kind"] == "transfers":
        return _exact_transfers(case, seed)
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed)
    if case["kind"] == "schemes" and case["scheme"] == "linear":
        return _exact_backtrack(case, seed)
    return None


def _exact_backtrack(case, seed):
    s = prepare(case, seed)
    D = s.p.D
    nodes = tuple(m + 1 for m in s.p.ni)
    ax = [_axis(a) for a in s.xv]
    grid = [[_axis(a) for a in g] for g in s.xi]
    mesh = torch.meshgrid(*[a[0] for a in reversed(ax)], indexing="ij")
    x = [m.reshape(-1) for m in reversed(mesh)]
    inner = torch.ones(mesh[0].shape, dtype=torch.bool, device="cuda")
    for d in range(D):
        at = [slice(None)] * D
        for end in (0, nodes[D - 1 - d] - 1):
            at[d] = end
            inner[tuple(at)] = False
    inner = inner.reshape(-1)
    x = [v[inner] for v in x]
    V = [_view(v) for v in s.V]
    k1 = _velocity(grid, V, x)
    if case["method"] == "rk2":
        al = case["alpha"]
        k2 = _velocity(grid, V, [a - al * s.dt * k for a, k in zip(x, k1)])
        b = 0.5 / al
        x = [a - s.dt * ((1.0 - b) * p + b * q) for a, p, q in zip(x, k1, k2)]
    else:
        k2 = _velocity(grid, V, [a - 0.5 * s.dt * k for a, k in zip(x, k1)])
        k3 = _velocity(grid, V, [a - 0.5 * s.dt * k for a, k in zip(x, k2)])
        k4 = _velocity(grid, V, [a - s.dt * k for a, k in zip(x, k3)])
        x = [a - s.dt * (p + 2 * q + 2 * r + u) / 6 for a, p, q, r, u in zip(x, k1, k2, k3, k4)]
    idx = [_bracket(a[0], v) for a, v in zip(ax, x)]
    out = []
    for T0, T in zip(s.T0, s.T):
        # several fields take the spacing at the node, which a range grid does
        # not tell from the spacing at the cell
        if len(s.T) > 1 and case["axes"] == "vector":
            return None
        t = [(v - a[0][i]) / a[1][i] for v, a, i in zip(x, ax, idx)]
        f = _view(T).clone().reshape(-1)
        f[inner] = _lerp(_view(T0), idx, t)
        out.append(f.reshape(_view(T).shape))
    return {"coords": [None] * D, "index": None, "fields": [None] * len(s.Fp), "nodal": out}
