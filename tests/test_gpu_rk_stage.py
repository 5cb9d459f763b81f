"""Runge-Kutta stages taken in the cell launch against the launch of their own
that follows the fused face-cell launch: the same bits, at sizes around a
block and for single cases and batches."""
import numpy as np
import pytest

from tmp_amd import mesh as MM
from tmp_amd import usg

pytestmark = pytest.mark.gpu


def _run(make, fused):
    with make() as s:
        s.fused(fused)
        r = np.random.default_rng(4)
        U = s.U
        s.set_prim(U * (1.0 + 1e-2 * r.uniform(-1, 1, U.shape)))
        h = s.rk5(3, history=True)
        return h, s.U, s.field(usg.F_CONS), s.field(usg.F_W0), s.R


@pytest.mark.parametrize("flow", [usg.EULER, usg.LAMINAR], ids=["euler", "laminar"])
@pytest.mark.parametrize("ni,nj", [(1, 1), (15, 17), (16, 16), (257, 1), (90, 70)])
def test_stage_in_the_cell_launch(ni, nj, flow):
    m = MM.rect(ni, nj, jitter=0.1, seed=2, bottom=MM.WALL)
    kw = dict(flow=flow, mach=0.5, aoa=2.0, reynolds=5000.0)
    for make in (lambda: usg.Solver(m, **kw),
                 lambda: usg.BatchSolver([m, MM.rect(9, 8, bottom=MM.WALL)], **kw)):
        for a, b in zip(_run(make, False), _run(make, True)):
            assert np.array_equal(a, b)
