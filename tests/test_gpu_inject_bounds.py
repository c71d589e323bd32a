"""Injection where its neighbour search meets particles outside their cells'
boxes: new particles of a cell whose spacing exceeds the distance of its vertices
(a range axis carries its first spacing for every cell), of an earlier colour
than the cell that searches; and on grids of one cell in a dimension.  FP64 bit
for bit against the oracle (runs on an MI355X)."""
import ctypes as C

import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip import _abi
from justpic_hip.particles import DeviceAxis
from justpic_hip.grids import Axis, staggered_grid
from oracle import oracle as O

from test_gpu_inject_cells import cells_of
from test_gpu_parity import assert_field, assert_state_equal, to_dev

pytestmark = pytest.mark.gpu


def narrowing(n):
    """A range axis of n cells whose first cell is the widest by 2 to 1, or less."""
    w = np.where(np.arange(n) % 3 == 0, 2.0, np.where(np.arange(n) % 3 == 1, 1.0, 1.4))
    return Axis(np.concatenate([[0.0], np.cumsum(w)]) / w.sum(), "range")


def sparse(n, K, seed):
    """A particle or none per cell, inside the cell."""
    xv = tuple(narrowing(m) for m in n)
    hp = O.HostParticles(xv, K, staggered_grid(xv))
    rng = np.random.default_rng(seed)
    e = np.arange(hp.S)
    occ = (e < hp.C) & (rng.random(hp.S) < 0.6)
    I = np.unravel_index(e % hp.C, hp.ni, order="F")
    for d in range(hp.D):
        a, b = hp.xv[d].x[I[d]], hp.xv[d].x[I[d] + 1]
        hp.coords[d][:] = np.where(occ, a + rng.uniform(0.05, 0.95, hp.S) * (b - a), np.nan)
    hp.index[:] = occ
    fields = [np.where(occ, rng.random(hp.S), np.nan) for _ in range(3)]
    return hp, fields, rng


# (cells, slots, min_xcell, fields)
CASES = [((7, 8, 5), 16, 8, 1), ((7, 8, 5), 24, 16, 2), ((9, 14), 12, 4, 2), ((9, 14), 24, 16, 3),
         ((9, 14), 12, 4, 1)]


@pytest.mark.parametrize("n,K,mn,nf", CASES)
def test_new_particles_outside_their_cell(ctx, n, K, mn, nf):
    print("[gpu-inject-bounds]", n, K, mn, nf, flush=True)
    hp, fields, _ = sparse(n, K, seed=K + nf)
    p = to_dev(ctx, hp, min_xcell=mn, seed=5)
    fd = [cells_of(ctx, hp, a) for a in fields[:nf]]
    st = jp.inject_particles_(p, tuple(fd), stats=True)
    so = O.inject_particles(hp, fields[:nf], mn, 5, 0)
    assert st == so and so["injected"] > 0
    assert_state_equal(p, hp, exact=True)
    for a, b in zip(fd, fields):
        assert_field(a.data.flat(), b, exact=True)


@pytest.mark.parametrize("n,K,mn,nf", CASES)
def test_new_particles_outside_their_cell_phase(ctx, n, K, mn, nf):
    print("[gpu-inject-bounds] phase", n, K, mn, nf, flush=True)
    hp, fields, rng = sparse(n, K, seed=K + nf)
    phases = np.where(hp.index == 1, rng.integers(1, 9, hp.S), np.nan).astype(float)
    grids = [rng.random(tuple(m + 1 for m in n)) for _ in range(nf)]
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


@pytest.mark.parametrize("n,K,nf", [((1, 6), 12, 1), ((5, 1), 12, 2), ((1, 1), 8, 0), ((3, 1, 4), 16, 2),
                                    ((1, 4, 1), 16, 1)])
def test_phase_one_cell_thick(ctx, n, K, nf):
    """One cell in a dimension: no cell-centred field is possible and the centre axis
    has one point and no spacing; phases and nodal fields through the C interface."""
    print("[gpu-inject-bounds] thin", n, K, nf, flush=True)
    D, mn = len(n), 8
    xv = tuple(Axis.lin(0.0, 1.0 + d, m + 1) for d, m in enumerate(n))
    hp = O.HostParticles(xv, K)
    rng = np.random.default_rng(K + nf)
    e = np.arange(hp.S)
    occ = (e < 2 * hp.C) & (rng.random(hp.S) < 0.5)
    occ[0] = True
    I = np.unravel_index(e % hp.C, hp.ni, order="F")
    for d in range(D):
        u = rng.uniform(0.05, 0.95, hp.S)
        hp.coords[d][:] = np.where(occ, xv[d].x[I[d]] + u * xv[d].dx[I[d]], np.nan)
    hp.index[:] = occ
    phases = np.where(occ, rng.integers(1, 9, hp.S), np.nan).astype(float)
    fields = [np.where(occ, rng.random(hp.S), np.nan) for _ in range(nf)]
    grids = [rng.random(int(np.prod([m + 1 for m in n]))) for _ in range(nf)]
    cen = (C.c_int * max(1, nf))()

    def centres(arrays):  # x of every centre; spacings that no call has a use for
        return (_abi.jp_axis * D)(*[_abi.jp_axis(a, b, b, m) for (a, b), m in zip(arrays, n)])

    xc = [(a.x[:-1] + a.x[1:]) / 2 for a in xv]
    dc = [1.0 / a.dx for a in xv]

    axes = [DeviceAxis(ctx, a) for a in xv]
    grid = _abi.jp_cellgrid()
    grid.ndim, grid.max_xcell = D, K
    for d in range(D):
        grid.ni[d], grid.xv[d] = n[d], axes[d].abi()
    dx = [(jp.DeviceArray.from_host(ctx, a), jp.DeviceArray.from_host(ctx, b)) for a, b in zip(xc, dc)]
    dev = [cells_of(ctx, hp, a) for a in hp.coords + [phases] + fields]
    index = jp.CellArray(ctx, hp.ni, K, dtype=np.uint8)
    index.copy_from(hp.index)
    dg = [jp.DeviceArray.from_host(ctx, a) for a in grids]
    st = _abi.jp_stats()
    ctx.check(ctx.lib.jp_inject_particles_phase(
        ctx.h, C.byref(grid), centres([(a.ptr, b.ptr) for a, b in dx]),
        _abi.ptr_array([a.ptr for a in dev[:D]]), index.ptr, dev[D].ptr, nf,
        _abi.ptr_array([a.ptr for a in dev[D + 1:]]), _abi.ptr_array([a.ptr for a in dg]), cen, mn,
        3, 0, C.byref(st)), "inject_particles_phase!")
    so = _abi.jp_stats()
    p = O._p
    assert O.lib().jpo_inject_particles_phase(
        C.byref(hp._grid), centres([(p(a), p(b)) for a, b in zip(xc, dc)]), hp.coord_ptrs(),
        p(hp.index), p(phases), nf, _abi.ptr_array([p(a) for a in fields]),
        _abi.ptr_array([p(a) for a in grids]), cen, mn, 3, 0, C.byref(so)) == 0
    assert st.as_dict() == so.as_dict() and so.injected > 0
    assert np.array_equal(index.data.flat(), hp.index)
    for a, b in zip(dev, hp.coords + [phases] + fields):
        assert_field(a.data.flat(), b, exact=True)


def nearest_copies(before, after, u, fields, n, K, h):
    """Values of the new particles' fields: colours in order, slots of a cell in order,
    each copied from its nearest particle (offsets u; neighbour cell, then slot, on
    equal distances).  Also how many of the sources lie outside their cell."""
    D, C_ = len(n), int(np.prod(n))
    act, u = before.copy(), [a.astype(np.float64) for a in u]
    out, outside = [f.copy() for f in fields], 0
    cells = np.stack(np.unravel_index(np.arange(C_), n, order="F"), 1)
    for col in range(2 ** D):
        odd = [(col >> (D - 1 - d)) & 1 for d in range(D)]
        for c in np.nonzero((cells % 2 == odd).all(1))[0]:
            for k in np.nonzero(after[c::C_] & ~before[c::C_])[0]:
                e = c + C_ * k
                src, best = -1, np.inf
                for nb in range(3 ** D):
                    o = [(nb // 3 ** d) % 3 - 1 for d in range(D)]
                    J = cells[c] + o
                    if (J < 0).any() or (J >= n).any():
                        continue
                    j = int(np.ravel_multi_index(J, n, order="F")) + C_ * np.arange(K)
                    s = 0.0
                    for d in range(D):
                        r = (o[d] + u[d][j] - u[d][e]) * h[d]
                        s = s + r * r
                    s = np.where(act[j] & ~np.isnan(s), np.sqrt(s), np.inf)
                    q = int(np.argmin(s))
                    if s[q] < best:
                        src, best = int(j[q]), s[q]
                if src >= 0:
                    outside += any(not 0 <= u[d][src] <= 1 for d in range(D))
                    for f in out:
                        f[e] = f[src]
                act[e] = True
    return out, outside


@pytest.mark.parametrize("n,K,mn,nf", [((7, 6, 5), 24, 14, 1), ((5, 4, 6), 40, 32, 2),
                                       ((13, 11), 20, 12, 2), ((9, 14), 64, 48, 3)])
def test_split_particles_outside_their_cell(ctx, n, K, mn, nf):
    """Split offsets up to two cells out (advected and not moved) and NaN."""
    print("[gpu-inject-bounds] split", n, K, mn, nf, flush=True)
    xv = tuple(Axis.lin(0.0, 1.0, m + 1) for m in n)
    hp = O.HostParticles(xv, K, staggered_grid(xv))
    rng = np.random.default_rng(K + nf)
    fill = rng.choice([0.0, 0.05, 0.3, 0.9], hp.C, p=[0.25, 0.3, 0.35, 0.1])
    occ = rng.random(hp.S) < fill[np.arange(hp.S) % hp.C]
    I = np.unravel_index(np.arange(hp.S) % hp.C, hp.ni, order="F")
    for d in range(hp.D):  # (any place inside the cell: the offsets are replaced below)
        hp.coords[d][:] = np.where(occ, xv[d].x[I[d]] + 0.5 * xv[d].dx[I[d]], np.nan)
    hp.index[:] = occ
    s = jp.to_split(to_dev(ctx, hp, min_xcell=mn, seed=5))
    for a in s.coords:
        u = rng.uniform(0.0, 1.0, hp.S) + rng.choice([0, 0, 0, -2, -1, 1, 2], hp.S)
        u = np.where(rng.random(hp.S) < 0.01, np.nan, u)
        a.copy_from(np.where(occ, u, np.nan).astype(np.float32))
    fields = [np.where(occ, rng.random(hp.S), np.nan) for _ in range(nf)]
    fd = [cells_of(ctx, hp, a) for a in fields]
    st = jp.inject_particles_(s, tuple(fd), stats=True)
    after = s.index.data.flat().astype(bool)
    assert st["injected"] == (after & ~occ).sum() > 0
    want, outside = nearest_copies(occ, after, [a.data.flat() for a in s.coords], fields, hp.ni, K,
                                   [a.dx[0] for a in xv])
    assert outside > 0
    for a, b in zip(fd, want):
        assert_field(a.data.flat(), b, exact=True)
