"""The transfers that take several slots of a cell per thread, on slot counts off
their chunks (8; 4 for the flip), ragged rows, sparse and empty slot planes and
several fields: bit for bit against the oracle; the split grid2particle against the
same interpolation in numpy (seven rounded lerps of two operations each, both
sides: 32 units of 2^-53 of the largest value).  Runs on an MI355X."""
import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip.grids import Axis, staggered_grid
from oracle import oracle as O

from helpers import host_particles
from test_gpu_parity import assert_field, to_dev
from test_gpu_transfers import field

pytestmark = pytest.mark.gpu


def state(n, K, keep, seed=3):
    """holes at random, slots up to the last; the last planes empty if keep < 0.5"""
    xv = tuple(Axis.lin(0.0, 1.0 + d, m + 1) for d, m in enumerate(n))
    xi = staggered_grid(xv)
    hp = host_particles(xv, xi, max(K, 2 ** len(n)), 1, seed=seed)
    rng = np.random.default_rng(seed)
    C = hp.C
    live = rng.random((K, C)) < keep
    if keep < 0.5:
        live[K // 2:] = False
    x = [np.full((K, C), np.nan) for _ in n]
    cells = np.unravel_index(np.arange(C), n, order="F")
    for d, ax in enumerate(xv):
        lo, h = ax.x[cells[d]], ax.dx[cells[d]]
        x[d][live] = (lo + h * rng.uniform(0.01, 0.99, (K, C)))[live]
    out = O.HostParticles(xv, K, xi)
    for d in range(len(n)):
        out.coords[d][:] = x[d].ravel()
    out.index[:] = live.ravel()
    return xv, xi, out


def cells(ctx, hp, arrays):
    out = []
    for a in arrays:
        ca = jp.CellArray(ctx, hp.ni, hp.K)
        ca.copy_from(a)
        out.append(ca)
    return out


def lerp(t, v):
    v = list(v)
    for d in range(len(t)):
        v = [(1.0 - t[d]) * a + t[d] * b for a, b in zip(v[::2], v[1::2])]
    return v[0]


@pytest.mark.parametrize("n,K,keep,nf", [
    ((65, 7), 13, 0.6, 2), ((64, 3), 8, 0.9, 1), ((2, 2), 1, 0.9, 1), ((70, 5), 64, 0.3, 3),
    ((5, 9, 4), 11, 0.6, 2), ((66, 3, 2), 64, 0.5, 1), ((7, 2, 3), 20, 0.02, 2),
])
def test_transfers_match_oracle(ctx, n, K, keep, nf):
    print("[gpu-transfer-slots]", n, K, keep, nf, flush=True)
    xv, xi, hp = state(n, K, keep)
    p = to_dev(ctx, hp)
    rng = np.random.default_rng(1)
    on = hp.index == 1
    F = [field(xv, 1 + f) for f in range(nf)]
    F0 = [field(xv, 7 + f) for f in range(nf)]
    Fd = [jp.DeviceArray.from_host(ctx, f) for f in F]

    g = cells(ctx, hp, [np.full(hp.S, -2.0)])[0]
    jp.grid2particle_(g, Fd[0], p)
    assert_field(g.data.flat(), O.grid2particle(hp, F[0], np.full(hp.S, -2.0)), exact=True)

    Fp = [np.where(on, rng.random(hp.S), -5.0) for _ in range(nf)]
    Fpd = cells(ctx, hp, Fp)
    jp.grid2particle_flip_(tuple(Fpd), tuple(Fd),
                           tuple(jp.DeviceArray.from_host(ctx, f) for f in F0), p, alpha=0.3)
    O.grid2particle_flip(hp, Fp, F, F0, 0.3)
    for a, b in zip(Fpd, Fp):
        assert_field(a.data.flat(), b, exact=True)

    Cd = [jp.centroid_field(p, fill=-3.0) for _ in range(nf)]
    jp.particle2centroid_(tuple(Cd), tuple(Fpd), p)
    for a, b in zip(Cd, O.particle2centroid(hp, Fp, tuple_method=True)):
        assert_field(a.flat(), b, exact=True)

    xc = O.centre_axes(hp)
    G = [field(xc, 3 + f) for f in range(nf)]
    Gpd = cells(ctx, hp, [np.full(hp.S, -1.0) for _ in range(nf)])
    jp.centroid2particle_(tuple(Gpd), tuple(jp.DeviceArray.from_host(ctx, f) for f in G), p)
    Gp = [np.full(hp.S, -1.0) for _ in range(nf)]
    O.centroid2particle(hp, Gp, G)
    for a, b in zip(Gpd, Gp):
        assert np.array_equal(a.data.flat(), b)

    s = jp.to_split(p)
    g = cells(ctx, hp, [np.full(hp.S, -2.0)])[0]
    jp.grid2particle_(g, Fd[0], s)
    got = g.data.flat()
    assert np.all(got[~on] == -2.0)
    e = np.nonzero(on)[0]
    I = np.unravel_index(e % hp.C, n, order="F")
    t = [s.off[d].data.flat()[e].astype(np.float64) for d in range(len(n))]
    v = [F[0][tuple(I[d] + ((q >> d) & 1) for d in range(len(n)))] for q in range(2 ** len(n))]
    assert np.all(np.abs(got[e] - lerp(t, v)) <= 32 * 2.0 ** -53 * np.max(np.abs(F[0])))
