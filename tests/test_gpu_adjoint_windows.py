"""The LDS windows of the 2D adjoint kernels against the oracle (runs on an
MI355X): windows that hold tile and velocities, only the tile, or nothing (a
shuffled list touches the whole grid), lists shorter than a wavefront and over
several workgroups, steps whose points leave the window (CFL 6 around the
vortex), fewer steps than a checkpoint interval, refined axes, particles on
velocity nodes, every integrator.  Forward, x0bar and Tpbar bit for bit; Vbar
within 1e-12 of its largest magnitude (FP64 atomic adds, whose order varies), as
for the other adjoint tests."""
import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip.grids import staggered_grid
from oracle import oracle as O

from helpers import blob, cfl_dt, host_particles, sample
from test_gpu_adjoint import EULER, RK2, RK4, close_to, container, integrator
from test_gpu_advect_windows import refined

pytestmark = pytest.mark.gpu

# n, axes, method, alpha, CFL, steps, every, particles kept, order
CASES = [
    ((60, 50), "lin", RK2, 0.5, 0.7, 23, 10, None, "patches"),
    ((60, 50), "lin", RK2, 0.3, 0.7, 9, 4, None, "shuffled"),
    ((95, 83), "lin", RK2, 0.5, 0.7, 7, 3, None, "shuffled"),
    ((130, 97), "lin", RK4, 0.5, 0.7, 5, 2, None, "shuffled"),
    ((70, 41), "lin", RK2, 0.5, 6.0, 12, 4, None, "patches"),
    ((70, 41), "lin", EULER, 0.5, 0.9, 6, 10, None, "patches"),
    ((70, 41), "steep", RK2, 0.5, 0.9, 11, 5, None, "patches"),
    ((33, 64), "alternating", RK4, 0.5, 0.9, 8, 3, None, "patches"),
    ((2, 2), "lin", RK2, 0.5, 0.3, 3, 1, None, "patches"),
    ((64, 64), "lin", RK2, 0.5, 0.7, 11, 10, 1, "patches"),
    ((64, 64), "lin", RK2, 0.5, 0.7, 11, 10, 65, "shuffled"),
    ((400, 380), "lin", RK2, 0.5, 0.7, 6, 3, None, "patches"),
]


@pytest.mark.parametrize("n,how,method,alpha,cfl,steps,every,keep,order", CASES)
def test_windows_match_oracle(ctx, n, how, method, alpha, cfl, steps, every, keep, order):
    print("[gpu-adjoint-windows]", n, how, method, cfl, steps, every, keep, order, flush=True)
    xv = tuple(refined(m, how) for m in n)
    xi = staggered_grid(xv)
    V = tuple(sample(f, xi[c]) for c, f in enumerate((
        lambda x, y: 3.0 * np.sin(np.pi * x) * np.cos(np.pi * y),
        lambda x, y: -3.0 * np.cos(np.pi * x) * np.sin(np.pi * y))))
    hp = host_particles(xv, xi, 4, 1, seed=5)
    dt = cfl * cfl_dt(xv, V)
    m = hp.index.astype(bool)
    x0 = [c[m].copy() for c in hp.coords]
    rng = np.random.default_rng(9)
    x0[1][rng.random(x0[1].size) < 0.01] = xi[0][1].x[1]  # velocity node lines
    x0[0][rng.random(x0[0].size) < 0.01] = xi[1][0].x[n[0] // 2]
    if order == "shuffled":
        p = rng.permutation(x0[0].size)
        x0 = [np.ascontiguousarray(a[p]) for a in x0]
    x0 = [np.ascontiguousarray(a[:keep]) for a in x0]
    Tp = blob(x0)
    r = O.adjoint_forward(hp, V, method, alpha, dt, steps, x0, Tp, every=every)
    op = jp.AdvectionP2G(container(ctx, hp), integrator(method, alpha), dt, steps, every)
    F = op.forward(V, x0, Tp)
    assert np.array_equal(op.alive.flat()[:Tp.size], r["alive"])
    for d in range(2):
        assert np.array_equal(op.xN[d].flat()[:Tp.size], r["xN"][d], equal_nan=True)
    ck = op._fw["ckpt"].flat()[:r["ckpt"].size].reshape(r["ckpt"].shape)
    assert np.array_equal(ck, r["ckpt"], equal_nan=True)
    assert np.array_equal(F.flat(), r["F"], equal_nan=True)
    assert np.array_equal(op.W.flat(), r["W"])

    Fb = rng.standard_normal(r["F"].size)
    Fb[~np.isfinite(r["F"])] = 0.0
    Vb, xb, Tb = O.adjoint_backward(hp, V, method, alpha, dt, steps, x0, Tp, r["F"], r["W"], Fb)
    gVb, gxb, gTb = op.pullback(Fb)
    for d in range(2):
        assert np.array_equal(gxb[d].flat()[:Tp.size], xb[d], equal_nan=True)
        assert close_to(gVb[d].to_host(), Vb[d], 1e-12)
    assert np.array_equal(gTb.flat()[:Tp.size], Tb, equal_nan=True)
