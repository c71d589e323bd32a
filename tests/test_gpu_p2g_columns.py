"""particle2grid! in FP64 at the sizes where the node columns change (one node
per thread up to 16), with ragged ends, one to five fields, particles on nodes,
distances whose squares leave the fast weights' range, and empty cells, bit for
bit against the oracle (runs on an MI355X)."""
import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip.grids import Axis, staggered_grid
from oracle import oracle as O

from test_gpu_parity import assert_field, to_dev

pytestmark = pytest.mark.gpu


def state(n, K, L, seed):
    """Random particles in about half the slots; a band of empty cells, one of
    full ones, and particles exactly on a vertex."""
    xv = tuple(Axis.lin(0.0, L, m + 1) for m in n)
    hp = O.HostParticles(xv, K, staggered_grid(xv))
    rng = np.random.default_rng(seed)
    cells = np.arange(hp.S) % hp.C
    I = np.stack(np.unravel_index(cells, hp.ni, order="F"), 0)
    occ = rng.random(hp.S) < np.where(I[1] < 2, 0.0, np.where(I[1] < 4, 1.0, 0.5))
    hp.index[:] = occ
    on = rng.random(hp.S) < 0.002
    for d in range(hp.D):
        h = xv[d].x[1] - xv[d].x[0]
        x = xv[d].x[I[d]] + np.where(on, 0.0, rng.random(hp.S)) * h
        hp.coords[d][:] = np.where(occ, x, np.nan)
    return hp, [np.where(occ, rng.random(hp.S) - 0.3, np.nan) for _ in range(5)]


CASES = [
    # (cells, slots, domain length, fields)
    ((5, 9), 7, 1.0, 1),         # one node per thread, K not a multiple of 4
    ((257, 301), 6, 1.0, 2),     # 2 nodes
    ((401, 397), 5, 1.0, 3),     # 4, ragged end
    ((601, 499), 4, 1.0, 4),     # 8, two launches
    ((901, 803), 4, 1.0, 1),     # 16
    ((33, 29), 64, 1.0, 5),      # full occupancy words
    ((40, 37), 8, 1e-150, 2),    # squares below the range (and denormal)
    ((40, 37), 8, 1e-155, 1),
    ((40, 37), 8, 1e150, 2),     # above it
    ((7, 6, 5), 9, 1.0, 2),      # 3D, odd number of nodes along y
    ((47, 52, 33), 5, 1.0, 3),   # 3D, 2 nodes
    ((65, 64, 71), 4, 1.0, 1),   # 3D, 4 nodes
]


@pytest.mark.parametrize("n,K,L,nf", CASES)
def test_p2g_columns(ctx, n, K, L, nf):
    print("[gpu-p2g-columns]", n, K, L, nf, flush=True)
    hp, Fp = state(n, K, L, seed=nf + K)
    p = to_dev(ctx, hp)
    Fpd = []
    for a in Fp[:nf]:
        ca = jp.CellArray(ctx, hp.ni, hp.K)
        ca.copy_from(a)
        Fpd.append(ca)
    F = tuple(jp.nodal_field(p) for _ in range(nf))
    if nf == 1:
        jp.particle2grid_(F[0], Fpd[0], p)
        want = [O.particle2grid(hp, Fp[0])]
    else:
        jp.particle2grid_(F, tuple(Fpd), p)
        want = O.particle2grid_multi(hp, Fp[:nf])
    for f, b in zip(F, want):
        assert_field(f.flat(), b, exact=True)
