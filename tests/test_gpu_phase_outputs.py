"""update_phase_ratios! with some outputs left out (NULL): the kinds of locations
share one launch; those asked for equal the oracle bit for bit, the others are not
written.  Grids of a few cells and of ragged workgroups.  Runs on an MI355X."""
import numpy as np
import pytest

import justpic_hip as jp
from justpic_hip import _abi
from justpic_hip.grids import Axis, staggered_grid
from oracle import oracle as O

from helpers import host_particles
from test_gpu_parity import to_dev
from test_gpu_phases import dev_cells

pytestmark = pytest.mark.gpu

FACES = ("Vx", "Vy", "Vz")


@pytest.mark.parametrize("n,nph,ask", [
    ((40, 7), 3, ("center",)), ((40, 7), 6, ("vertex",)), ((16, 16), 2, ("Vy",)),
    ((33, 8), 4, ("Vx", "center")), ((2, 9), 3, ("vertex", "Vx", "Vy", "center")), ((9, 4), 2, ()),
    ((5, 6, 4), 3, ("Vz", "vertex")), ((4, 3, 9), 9, ("Vx", "Vy", "center")),
])
def test_outputs_left_out(ctx, n, nph, ask):
    print("[gpu-phase-outputs]", n, nph, ask, flush=True)
    D = len(n)
    xv = tuple(Axis.lin(0.0, 1.0 + 0.5 * d, m + 1) for d, m in enumerate(n))
    hp = host_particles(xv, staggered_grid(xv), 16 if D == 2 else 24, 2, seed=4)
    rng = np.random.default_rng(nph)
    phases = np.where(hp.index == 1, rng.integers(1, nph + 1, hp.S), np.nan).astype(float)
    want = O.update_phase_ratios(hp, phases, nph)
    p = to_dev(ctx, hp)
    pr = jp.PhaseRatios(ctx, nph, hp.ni)
    mark = {}
    for k, f in pr.fields.items():
        mark[k] = np.full(f.to_host().shape, -7.0)
        f.copy_from(mark[k])
    ptr = {k: (pr.fields[k].ptr if k in ask else None) for k in ("center", "vertex") + FACES[:D]}
    ph = dev_cells(ctx, hp, phases)
    ctx.check(ctx.lib.jp_update_phase_ratios(
        ctx.h, p.grid_ref(), p.centre_axes_ref(), p.coord_ptrs(), ph.ptr, nph, ptr["center"],
        ptr["vertex"], _abi.ptr_array([ptr[k] for k in FACES[:D]]), None), "update_phase_ratios!")
    for k in want:
        got = pr.fields[k].to_host()
        assert np.array_equal(got, want[k] if k in ask else mark[k], equal_nan=True), k
