"""FP64 advection on both sides of the rule that gives MQS and LinP a thread per slot
on small grids, and the tiled kernel's pass over the particles that leave the
windows: none, some and all of a wavefront, in containers whose slots are all, half
and hardly filled; split advection with the same steps against its own path without
windows.  Bit for bit (runs on an MI355X)."""
import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip.grids import staggered_grid
from oracle import oracle as O

from helpers import host_particles, sample
import test_gpu_split_windows as split_windows
from test_gpu_advect_windows import ADVECT, METHODS, refined, slots
from test_gpu_parity import assert_state_equal, dev_V, to_dev

pytestmark = pytest.mark.gpu


def state(n, K, npq, how, seed, patch):
    """Particles in every cell; velocities of one size, or (patch) much larger in a
    part of the grid, so that some wavefronts' particles all leave the windows and
    some wavefronts' only here and there."""
    xv = tuple(refined(m, how) for m in n)
    xi = staggered_grid(xv)
    D = len(n)
    rng = np.random.default_rng(seed)
    V = []
    for c in range(D):
        k = rng.uniform(1.0, 3.0, D)
        V.append(sample(lambda *X: np.prod([np.cos(k[d] * X[d] + c) for d in range(D)], 0) *
                        np.sin(np.pi * X[c]) *
                        (np.where(X[0] > 0.6, 8.0, 0.9) if patch else 1.0), xi[c]))
    hp = host_particles(xv, xi, K, npq, seed=seed)
    gone = rng.random(hp.S) < 0.2  # holes, so that the lanes' counts differ
    hp.index[gone] = 0
    for c in hp.coords:
        c[gone] = np.nan
    return xv, V, hp


# cells, slots, per quadrant, axes, CFL, patch; 2D: 64 * ceil(nx / 64) * ny slots a plane
CASES = [
    ((131, 60), 64, 6, "uniform", 0.9, False),   # tiles
    ((131, 60), 64, 12, "smooth", 0.9, True),
    ((70, 90), 64, 14, "alternating", 6.0, False),
    ((256, 54), 48, 3, "uniform", 6.0, True),
    ((131, 53), 64, 6, "uniform", 0.9, True),    # 10176 wavefronts of slots
    ((33, 20, 20), 32, 3, "uniform", 0.9, True),
    ((18, 30, 21), 24, 2, "smooth", 5.0, False),
    ((17, 19, 13), 40, 2, "steep", 0.9, True),   # 9880
]


@pytest.mark.parametrize("scheme", ["linear", "MQS", "LinP"])
@pytest.mark.parametrize("method", ["rk2", "rk4"])
@pytest.mark.parametrize("n,K,npq,how,cfl,patch", CASES)
def test_routes(ctx, n, K, npq, how, cfl, patch, method, scheme):
    print("[gpu-advect-routes]", n, K, npq, how, cfl, patch, method, scheme, flush=True)
    xv, V, hp = state(n, K, npq, how, K + n[0], patch)
    dt = cfl * min(np.min(a.dx) for a in xv) / max(np.abs(v).max() for v in V)
    if patch:
        dt *= 8.0 / 0.9
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


@pytest.mark.parametrize("n,K,keep,how,method,cfl", [
    ((64, 64), 48, 0.5, "std", "rk4", 8.0),
    ((130, 17), 64, 0.9, "std", "rk2", 6.0),
    ((70, 33), 24, 0.3, "ghosts", "rk4", 1.6),
    ((200, 5), 64, 0.9, "std", "rk2w", 2.0),
    ((33, 9, 5), 64, 0.5, "std", "rk4", 6.0),
    ((16, 8, 12), 54, 0.5, "std", "rk2", 2.0),
])
def test_split_far_steps(ctx, n, K, keep, how, method, cfl):
    split_windows.test_windows_equal_global(ctx, n, K, keep, how, method, cfl)
