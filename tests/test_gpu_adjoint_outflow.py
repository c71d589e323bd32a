"""The adjoint's forward pass with particles carried out of the grid, in lists of
several workgroups (runs on an MI355X): stage points just outside a component's
grid, far outside and infinite (the stages after the first +Inf of RK2 and RK4), on
the boundary itself, beside points of the same wavefront that stay inside; uniform
and refined axes, with windows and without (a shuffled list).  Survivors, final
positions, checkpoints, F and W bit for bit against the oracle; x0bar and Tpbar of
the survivors too, Vbar within 1e-12 of its largest magnitude (FP64 atomic adds,
whose order varies)."""
import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip.grids import staggered_grid
from oracle import oracle as O

from helpers import blob, cfl_dt, host_particles, sample
from test_gpu_adjoint import EULER, RK2, RK4, close_to, container, integrator
from test_gpu_advect_windows import refined

pytestmark = pytest.mark.gpu

# n, axes, method, alpha, CFL, steps, every, order
CASES = [
    ((60, 50), "lin", RK2, 0.5, 0.7, 17, 4, "patches"),
    ((60, 50), "lin", RK4, 0.5, 0.7, 17, 4, "patches"),
    ((60, 50), "lin", EULER, 0.5, 0.9, 9, 4, "patches"),
    ((95, 83), "lin", RK4, 0.5, 0.9, 9, 3, "shuffled"),
    ((60, 50), "lin", RK2, 0.3, 7.0, 5, 2, "patches"),
    ((60, 50), "lin", RK4, 0.5, 90.0, 3, 2, "patches"),
    ((33, 64), "steep", RK4, 0.5, 0.9, 12, 5, "patches"),
    ((12, 9, 10), "lin", RK2, 0.5, 0.7, 7, 3, "patches"),
    ((12, 9, 10), "lin", RK4, 0.5, 0.7, 7, 3, "patches"),
    ((12, 9, 10), "alternating", RK4, 0.5, 6.0, 3, 2, "patches"),
]


@pytest.mark.parametrize("n,how,method,alpha,cfl,steps,every,order", CASES)
def test_outflow_matches_oracle(ctx, n, how, method, alpha, cfl, steps, every, order):
    print("[gpu-adjoint-outflow]", n, how, method, cfl, steps, every, order, flush=True)
    D = len(n)
    xv = tuple(refined(m, how) for m in n)
    xi = staggered_grid(xv)
    # through the grid, faster in the middle, with a part that turns
    V = tuple(sample(lambda *x, c=c: (3.0, 1.5, -0.8)[c] * (1.0 + 0.5 * np.sin(np.pi * x[1 - c % 2])) +
                     0.6 * np.sin(2 * np.pi * x[c]), xi[c]) for c in range(D))
    hp = host_particles(xv, xi, 8 if D == 2 else 16, 1, seed=5)
    dt = cfl * cfl_dt(xv, V)
    m = hp.index.astype(bool)
    x0 = [c[m].copy() for c in hp.coords]
    rng = np.random.default_rng(9)
    for d in range(D):  # on the first and last vertex
        x0[d][rng.random(x0[d].size) < 0.01] = xv[d].x[0]
        x0[d][rng.random(x0[d].size) < 0.01] = xv[d].x[-1]
    if order == "shuffled":
        p = rng.permutation(x0[0].size)
        x0 = [np.ascontiguousarray(a[p]) for a in x0]
    Tp = blob(x0)
    r = O.adjoint_forward(hp, V, method, alpha, dt, steps, x0, Tp, every=every)
    assert 0 < r["alive"].sum() < Tp.size or cfl > 50
    op = jp.AdvectionP2G(container(ctx, hp), integrator(method, alpha), dt, steps, every)
    F = op.forward(V, x0, Tp)
    assert np.array_equal(op.alive.flat()[:Tp.size], r["alive"])
    for d in range(D):
        assert np.array_equal(op.xN[d].flat()[:Tp.size], r["xN"][d], equal_nan=True)
    ck = op._fw["ckpt"].flat()[:r["ckpt"].size].reshape(r["ckpt"].shape)
    assert np.array_equal(ck, r["ckpt"], equal_nan=True)
    assert np.array_equal(F.flat(), r["F"], equal_nan=True)
    assert np.array_equal(op.W.flat(), r["W"])

    Fb = rng.standard_normal(r["F"].size)
    Fb[~np.isfinite(r["F"])] = 0.0
    Vb, xb, Tb = O.adjoint_backward(hp, V, method, alpha, dt, steps, x0, Tp, r["F"], r["W"], Fb)
    gVb, gxb, gTb = op.pullback(Fb)
    for d in range(D):
        assert np.array_equal(gxb[d].flat()[:Tp.size], xb[d], equal_nan=True)
        assert close_to(gVb[d].to_host(), Vb[d], 1e-12)
    assert np.array_equal(gTb.flat()[:Tp.size], Tb, equal_nan=True)
