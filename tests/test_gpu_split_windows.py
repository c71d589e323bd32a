"""The split advection's LDS windows against the same arithmetic from global
memory (the split forward of the adjoint, one step), bit for bit: tile edges and
ragged tiles, slots up to 64 with holes, few and no particles, standard and other
velocity axes, steps that leave the windows (CFL 2.7, or twice as many nodes as
cells) and the domain.  The grid spacing is a power of two, so that a position and
its offset convert exactly.  Runs on an MI355X."""
import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip.grids import Axis, staggered_grid

from helpers import host_particles, sample

pytestmark = pytest.mark.gpu

H = 1.0 / 32
METHODS = {"euler": jp.Euler(), "rk2": jp.RungeKutta2(), "rk2w": jp.RungeKutta2(0.7),
           "rk4": jp.RungeKutta4()}


def velocity_axes(xv, how):
    xi = [list(a) for a in staggered_grid(xv)]
    D = len(xv)
    for c in range(D):
        for d in range(D):
            n = xv[d].n - 1
            if how == "ghosts" and c != d:  # a second ghost centre
                xi[c][d] = Axis.lin(-1.5 * H, (n + 1.5) * H, n + 4)
            if how == "double" and c != d:  # two nodes per cell
                xi[c][d] = Axis((np.arange(2 * n + 3) - 1) * (H / 2))
    return tuple(tuple(a) for a in xi)


@pytest.mark.parametrize("n,K,keep,how,method,cfl", [
    ((64, 64), 24, 0.6, "std", "rk2", 1.0),
    ((67, 9), 64, 0.5, "std", "rk4", 1.0),
    ((130, 7), 20, 0.9, "std", "rk2w", 2.7),
    ((5, 3), 12, 0.1, "std", "euler", 0.4),
    ((40, 70), 33, 0.6, "ghosts", "rk4", 1.0),
    ((40, 21), 24, 0.6, "double", "rk2", 0.9),
    ((33, 9, 5), 64, 0.5, "std", "rk2", 1.0),
    ((31, 6, 7), 24, 0.7, "std", "rk4", 2.7),
    ((40, 5, 6), 24, 0.02, "ghosts", "rk2w", 1.0),
    ((12, 10, 8), 24, 0.6, "double", "euler", 1.0),
])
def test_windows_equal_global(ctx, n, K, keep, how, method, cfl):
    print("[gpu-split-windows]", n, K, keep, how, method, cfl, flush=True)
    D = len(n)
    xv = tuple(Axis(np.arange(m + 1) * H) for m in n)  # (exact; a linspace rounds)
    xi = velocity_axes(xv, how)
    rng = np.random.default_rng(17)
    k = rng.uniform(2.0, 5.0, (D, D))
    V = tuple(sample(lambda *X, c=c: np.prod([np.cos(k[c, d] * X[d] + c) for d in range(D)], 0),
                     xi[c]) for c in range(D))
    dt = cfl * H / max(np.max(np.abs(v)) for v in V)
    hp = host_particles(xv, xi, K, 2 if K < 40 or D == 3 else 3, seed=7)
    C = hp.C
    # holes, and slots up to the last one
    order = np.argsort(rng.random((K, C)), axis=0)
    drop = rng.random((K, C)) >= keep
    index = np.take_along_axis(hp.index.reshape(K, C), order, 0)
    index[drop] = 0
    for d in range(D):
        x = np.take_along_axis(hp.coords[d].reshape(K, C), order, 0)
        hp.coords[d][:] = np.where(index == 1, x, np.nan).ravel()
    hp.index[:] = index.ravel()
    p = jp.particles_from_host(ctx, xi, hp.coords, hp.index, K, K, 1)
    s = jp.to_split(p)
    e = np.nonzero(hp.index)[0]
    cells = np.unravel_index(e % C, n, order="F")
    u0 = [s.off[d].data.flat()[e] for d in range(D)]
    x0 = [np.ascontiguousarray(cells[d] * H + u0[d].astype(np.float64) * H) for d in range(D)]
    dV = tuple(jp.DeviceArray.from_host(ctx, v) for v in V)
    jp.advection_(s, METHODS[method], dV, dt)
    out = [s.off[d].data.flat() for d in range(D)]
    assert all(np.all(np.isnan(o[hp.index == 0])) for o in out)
    out = [o[e] for o in out]

    op = jp.AdvectionP2G(p, METHODS[method], dt, 1, 1, form="split")
    op.forward(dV, x0, np.ones(e.size))
    fin = np.all([np.abs(o) < 1.0e6 for o in out], 0)
    sd = [np.where(fin, np.floor(np.where(fin, o, 0.0)), 0).astype(np.int64) for o in out]
    J = [c + a for c, a in zip(cells, sd)]
    here = fin & np.all([(j >= 0) & (j < m) for j, m in zip(J, n)], 0)
    assert np.array_equal(op.alive.flat()[:e.size].astype(bool), here)
    assert here.any() or e.size == 0
    for d in range(D):
        u = (out[d].astype(np.float64) - sd[d]).astype(np.float32)
        x = np.where(here, J[d] * H + u.astype(np.float64) * H,
                     cells[d] * H + out[d].astype(np.float64) * H)
        assert np.array_equal(op.xN[d].flat()[:e.size], x, equal_nan=True)
