"""Both sides of the grid-to-particle kernels' choice of 2 or 8 slots of a cell per
thread (8 from 12 wavefronts per CU on: 3072 of 8 slots on 256 CUs), on slot counts
off both chunks, ragged rows, the sizes next to the line: grid2particle and
centroid2particle bit for bit against the oracle, the split grid2particle against the
same interpolation in numpy (seven rounded lerps of two operations each, both sides:
32 units of 2^-53 of the largest value).  Runs on an MI355X."""
import numpy as np
import pytest

import justpic_hip as jp
from oracle import oracle as O

from test_gpu_parity import assert_field, to_dev
from test_gpu_transfer_slots import cells, lerp, state
from test_gpu_transfers import field

pytestmark = pytest.mark.gpu


def waves(n, K):
    return -(-n[0] // 64) * int(np.prod(n[1:])) * -(-K // 8)


@pytest.mark.parametrize("n,K,keep,over", [
    ((70, 511), 23, 0.6, False), ((70, 512), 23, 0.6, True),       # 3066, 3072
    ((130, 127), 63, 0.3, False), ((130, 129), 63, 0.9, True),     # 3048, 3096
    ((20, 60, 25), 13, 0.6, False), ((20, 60, 27), 13, 0.6, True),  # 3000, 3240
])
def test_both_sides_match(ctx, n, K, keep, over):
    print("[gpu-slots-per-thread]", n, K, keep, over, flush=True)
    assert (waves(n, K) >= 12 * 256) == over
    xv, xi, hp = state(n, K, keep)
    p = to_dev(ctx, hp)
    on = hp.index == 1
    F = field(xv, 1)
    Fd = jp.DeviceArray.from_host(ctx, F)

    g = cells(ctx, hp, [np.full(hp.S, -2.0)])[0]
    jp.grid2particle_(g, Fd, p)
    assert_field(g.data.flat(), O.grid2particle(hp, F, np.full(hp.S, -2.0)), exact=True)

    G = [field(O.centre_axes(hp), 3 + f) for f in range(2)]
    Gpd = cells(ctx, hp, [np.full(hp.S, -1.0) for _ in G])
    jp.centroid2particle_(tuple(Gpd), tuple(jp.DeviceArray.from_host(ctx, f) for f in G), p)
    Gp = [np.full(hp.S, -1.0) for _ in G]
    O.centroid2particle(hp, Gp, G)
    for a, b in zip(Gpd, Gp):
        assert np.array_equal(a.data.flat(), b)

    s = jp.to_split(p)
    g = cells(ctx, hp, [np.full(hp.S, -2.0)])[0]
    jp.grid2particle_(g, Fd, s)
    got = g.data.flat()
    assert np.all(got[~on] == -2.0)
    e = np.nonzero(on)[0]
    I = np.unravel_index(e % hp.C, n, order="F")
    t = [s.off[d].data.flat()[e].astype(np.float64) for d in range(len(n))]
    v = [F[tuple(I[d] + ((q >> d) & 1) for d in range(len(n)))] for q in range(2 ** len(n))]
    assert np.all(np.abs(got[e] - lerp(t, v)) <= 32 * 2.0 ** -53 * np.max(np.abs(F)))
