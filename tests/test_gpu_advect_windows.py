"""MQS and LinP advection from the LDS windows of the tiled kernel, and the
windows on refined axes (brackets searched from the particle's cell), at tile
edges, grids smaller than a window, steps beyond the windows and particles on
velocity nodes, bit for bit against the oracle and the slot kernel (runs on an
MI355X)."""
import contextlib

import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip import _abi
from justpic_hip.grids import Axis, staggered_grid
from oracle import oracle as O

from helpers import host_particles, sample
from test_gpu_parity import assert_state_equal, dev_V, to_dev

pytestmark = pytest.mark.gpu

ADVECT = {"linear": jp.advection_, "MQS": jp.advection_MQS_, "LinP": jp.advection_LinP_}
METHODS = {"rk2": (jp.RungeKutta2(), O.JP_RK2), "rk4": (jp.RungeKutta4(), O.JP_RK4),
           "euler": (jp.Euler(), O.JP_EULER)}


@contextlib.contextmanager
def slots(ctx):
    ctx.set_option(_abi.JP_OPT_ADVECT_SLOTS, 1)
    try:
        yield
    finally:
        ctx.set_option(_abi.JP_OPT_ADVECT_SLOTS, 0)


def refined(n, how):
    x = np.linspace(0.0, 1.0, n + 1)
    if how == "smooth":  # towards the middle
        return Axis(x + 0.25 * np.sin(2 * np.pi * x) / (2 * np.pi), "vector")
    if how == "steep":  # towards one end, 1 to 20
        return Axis((np.exp(3.0 * x) - 1.0) / (np.exp(3.0) - 1.0), "vector")
    if how == "alternating":  # neighbouring cells of different width
        d = np.where(np.arange(n) % 2 == 0, 1.0, 2.5)
        return Axis(np.concatenate([[0.0], np.cumsum(d)]) / d.sum(), "vector")
    return Axis.lin(0.0, 1.0, n + 1)


def state(n, how, seed):
    xv = tuple(refined(m, how) for m in n)
    xi = staggered_grid(xv)
    D = len(n)
    rng = np.random.default_rng(seed)
    V = []
    for c in range(D):
        k = rng.uniform(1.0, 3.0, D)
        V.append(sample(lambda *X: np.prod([np.cos(k[d] * X[d] + c) for d in range(D)], 0) *
                        np.sin(np.pi * X[c]), xi[c]))
    hp = host_particles(xv, xi, 10 if D == 2 else 12, 2 if D == 2 else 1, seed=seed)
    # some particles on a velocity node line
    on = rng.random(hp.S) < 0.02
    nodes = xi[0][1].x
    y = hp.coords[1]
    k = np.clip(np.searchsorted(nodes, np.nan_to_num(y)), 1, nodes.size - 2)
    inside = on & (hp.index == 1) & (nodes[k] > xv[1].x[0]) & (nodes[k] < xv[1].x[-1])
    y[inside] = nodes[k][inside]
    return xv, xi, V, hp


@pytest.mark.parametrize("scheme", ["linear", "MQS", "LinP"])
@pytest.mark.parametrize("n,how,method,cfl", [
    ((131, 11), "uniform", "rk4", 0.9),
    ((131, 11), "smooth", "rk2", 0.9),
    ((70, 9), "steep", "rk4", 0.8),
    ((65, 5), "alternating", "rk2", 0.9),
    ((3, 4), "smooth", "rk4", 0.5),
    ((130, 9), "smooth", "rk2", 6.0),
    ((18, 9, 6), "uniform", "rk2", 0.9),
    ((33, 7, 5), "smooth", "rk4", 0.9),
    ((17, 5, 9), "steep", "euler", 0.8),
    ((20, 6, 5), "smooth", "rk2", 5.0),
])
def test_windows(ctx, n, how, method, cfl, scheme):
    print("[gpu-advect-windows]", n, how, method, cfl, scheme, flush=True)
    xv, xi, V, hp = state(n, how, seed=len(n) * 10 + n[0])
    dt = cfl * min(np.min(a.dx) for a in xv) / max(np.abs(v).max() for v in V)
    rk, code = METHODS[method]
    p, q = to_dev(ctx, hp), to_dev(ctx, hp)
    Vd = dev_V(ctx, V)
    ADVECT[scheme](p, rk, Vd, dt)
    with slots(ctx):
        ADVECT[scheme](q, rk, Vd, dt)
    if scheme == "linear":
        O.advection(hp, V, code, 0.5, dt)
    else:
        O.advection_scheme(hp, V, code, 0.5, dt, scheme)
    assert_state_equal(q, hp, exact=True)
    assert_state_equal(p, hp, exact=True)
