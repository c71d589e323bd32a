"""Injection in 3D, with several fields and with phases, where the neighbour
search's pruning, its order and its rounds can go wrong: particles outside their
cells' boxes (advected and not moved, NaN coordinates), empty and crowded
neighbourhoods, more than 16 injections in one cell, equal distances (a dyadic
lattice), one to five fields, K = 64, refined axes; FP64 bit for bit against the
oracle, the split form with the same masks, copies and counts (runs on an
MI355X)."""
import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip.grids import Axis, staggered_grid
from oracle import oracle as O

from test_gpu_parity import assert_field, assert_state_equal, to_dev

pytestmark = pytest.mark.gpu


def axis(n, refined):
    if not refined:
        return Axis(np.arange(n + 1) / n, "range")
    x = np.linspace(0.0, 1.0, n + 1)
    return Axis(x + 0.3 * np.sin(2 * np.pi * x) / (2 * np.pi), "vector")


def state(n, K, how, seed):
    """Uneven cells (empty to full); how: `spread` particles may lie up to two
    cells away from their slot's cell, `lattice` on multiples of 1/8 cell."""
    xv = tuple(axis(m, how == "refined") for m in n)
    hp = O.HostParticles(xv, K, staggered_grid(xv))
    rng = np.random.default_rng(seed)
    cells = np.arange(hp.S) % hp.C
    fill = rng.choice([0.0, 0.05, 0.3, 0.9], hp.C, p=[0.25, 0.3, 0.35, 0.1])
    if how == "lonely":
        fill[:] = 0.0
        fill[rng.integers(0, hp.C, 2)] = 0.1
    occ = rng.random(hp.S) < fill[cells]
    I = np.stack(np.unravel_index(cells, hp.ni, order="F"), 0)
    for d in range(hp.D):
        u = rng.uniform(0.01, 0.99, hp.S)
        if how == "lattice":
            u = rng.integers(1, 8, hp.S) / 8.0
        if how == "spread":
            u = u + rng.choice([0, 0, 0, -2, -1, 1, 2], hp.S)
        x = hp.xv[d].x[I[d]] + u * hp.xv[d].dx[np.minimum(I[d], hp.ni[d] - 1)]
        if how == "spread":
            x = np.where(rng.random(hp.S) < 0.01, np.nan, x)
        hp.coords[d][:] = np.where(occ, x, np.nan)
    hp.index[:] = occ
    fields = [np.where(occ, rng.random(hp.S), np.nan) for _ in range(5)]
    return hp, fields, rng


def cells_of(ctx, hp, a):
    ca = jp.CellArray(ctx, hp.ni, hp.K)
    ca.copy_from(a)
    return ca


CASES = [
    # (cells, slots, min_xcell, fields, state)
    ((7, 6, 5), 24, 14, 1, "even"),
    ((7, 6, 5), 40, 32, 2, "even"),      # up to 32 injections in a cell
    ((6, 5, 7), 64, 60, 3, "even"),      # up to 64
    ((6, 5, 4), 10, 16, 1, "lattice"),
    ((8, 5, 6), 20, 16, 2, "spread"),
    ((5, 5, 5), 16, 16, 1, "lonely"),
    ((6, 7, 5), 18, 16, 5, "refined"),
    ((2, 2, 2), 12, 8, 0, "even"),
    ((19, 14), 24, 12, 2, "even"),
    ((19, 14), 64, 48, 5, "even"),
    ((16, 8), 12, 8, 2, "lattice"),
    ((15, 13), 20, 12, 3, "spread"),
    ((2, 3), 12, 8, 2, "refined"),
]


@pytest.mark.parametrize("n,K,mn,nf,how", CASES)
def test_inject_cells(ctx, n, K, mn, nf, how):
    print("[gpu-inject-cells]", n, K, mn, nf, how, flush=True)
    hp, fields, _ = state(n, K, how, seed=K + nf)
    p = to_dev(ctx, hp, min_xcell=mn, seed=5)
    fd = [cells_of(ctx, hp, a) for a in fields[:nf]]
    st = jp.inject_particles_(p, tuple(fd), stats=True)
    so = O.inject_particles(hp, fields[:nf], mn, 5, 0)
    assert st == so and so["injected"] > 0
    assert_state_equal(p, hp, exact=True)
    for a, b in zip(fd, fields):
        assert_field(a.data.flat(), b, exact=True)


@pytest.mark.parametrize("n,K,mn,nf,how", [c for c in CASES if c[3] < 5])
def test_inject_cells_phase(ctx, n, K, mn, nf, how):
    print("[gpu-inject-cells] phase", n, K, mn, nf, how, flush=True)
    hp, fields, rng = state(n, K, how, seed=K + nf)
    phases = np.where(hp.index == 1, rng.integers(1, 4, hp.S), np.nan).astype(float)
    grids = [rng.random(tuple(m + (1 - a % 2) for m in n)) for a in range(nf)]
    p = to_dev(ctx, hp, min_xcell=mn, seed=9)
    ph = cells_of(ctx, hp, phases)
    fd = [cells_of(ctx, hp, a) for a in fields[:nf]]
    st = jp.inject_particles_phase_(p, ph, tuple(fd),
                                    tuple(jp.DeviceArray.from_host(ctx, g) for g in grids),
                                    stats=True)
    so = O.inject_particles_phase(hp, phases, fields[:nf], grids, mn, 9, 0)
    assert st == so and so["injected"] > 0
    assert_state_equal(p, hp, exact=True)
    assert_field(ph.data.flat(), phases, exact=True)
    for a, b in zip(fd, fields):
        assert_field(a.data.flat(), b, exact=True)


@pytest.mark.parametrize("n,K,mn,nf,how", [c for c in CASES if c[4] in ("even", "lattice")])
def test_inject_cells_split(ctx, n, K, mn, nf, how):
    """Positions at multiples of 1/64 of power-of-two cells are the same in both
    forms, so are the distances between them; new positions round to float32,
    so searches among them are left to chance (masks and counts are not)."""
    print("[gpu-inject-cells] split", n, K, mn, nf, how, flush=True)
    n = tuple(1 << (m.bit_length() - 1) for m in n)
    hp, fields, rng = state(n, K, "lattice", seed=K + nf)
    s = jp.to_split(to_dev(ctx, hp, min_xcell=mn, seed=5))
    fd = [cells_of(ctx, hp, a) for a in fields[:nf]]
    st = jp.inject_particles_(s, tuple(fd), stats=True)
    so = O.inject_particles(hp, fields[:nf], mn, 5, 0)
    assert st == so
    p = jp.to_f64(s)
    coords, index = p.host_state()
    assert np.array_equal(index, hp.index)
    m = hp.index == 1
    for d in range(hp.D):
        assert np.max(np.abs(coords[d][m] - hp.coords[d][m])) <= 2.0 ** -24 / n[d]
    for a, b in zip(fd, fields):
        same = a.data.flat()[m] == b[m]
        assert np.mean(same) > 0.995, np.mean(same)
