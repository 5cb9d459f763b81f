"""Sweeps of many narrow levels (k_levels): meshes in their file's or
generator's numbering, whose sweeps have more levels than the launch
threshold, against the oracle; a batch of such meshes against its single
cases; and blanked cells."""
import numpy as np
import pytest

from oracle import oracle as O
from tmp_amd import mesh, usg

from .common import part2

pytestmark = pytest.mark.gpu

# the trajectory bar of the parity tests: libm's last bits, carried over the steps
TOL = 1e-12

MESHES = {
    # 122 levels of at most 22 cells: one chunk each
    "part2": part2,
    # quads in row order, levels of one cell up to the short side
    "rows": lambda: mesh.rect(9, 40, jitter=0.1, seed=1, bottom=mesh.WALL),
    # levels of exactly a chunk (64 cells) and of one more, of a whole round of
    # four chunks and of one more
    "chunk": lambda: mesh.rect(64, 70, bottom=mesh.WALL),
    "chunk_and_one": lambda: mesh.rect(65, 70, bottom=mesh.WALL),
    "round": lambda: mesh.rect(256, 260, bottom=mesh.WALL),
    "round_and_one": lambda: mesh.rect(257, 260, bottom=mesh.WALL),
    # the widest narrow level, and levels one cell wider, which keep their launches
    "widest": lambda: mesh.rect(512, 515, bottom=mesh.WALL),
    "too_wide": lambda: mesh.rect(513, 515, bottom=mesh.WALL),
    # triangles and quads: three dependencies, and neighbours many levels back
    "hybrid": lambda: mesh.airfoil_hybrid(ni=64, dy1=1e-3, rfar=10.0),
}


@pytest.mark.parametrize("flow", [usg.EULER, usg.LAMINAR, usg.SST], ids=["euler", "laminar", "sst"])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_level_sweeps_match_oracle(name, flow):
    m = MESHES[name]()
    s = usg.Solver(m, flow=flow, mach=0.3, aoa=2.0, reynolds=1e4)
    assert sum(s.waves()) > 14
    o = O.OracleSolver(O.OracleMesh(m), flow, 0.3, 2.0, 1e4)
    h = s.lusgs(5, history=True)
    ref = []
    for _ in range(5):
        o.lusgs_step()
        ref.append(o.res_l2())
    err = np.max(np.abs(s.U - o.U), axis=0) / np.max(np.abs(o.U), axis=0)
    assert np.all(err <= TOL), err
    assert np.all(np.abs(h - ref) <= TOL * np.abs(ref))


@pytest.mark.parametrize("flow", [usg.EULER, usg.SST], ids=["euler", "sst"])
def test_level_sweeps_of_a_batch_equal_single_cases(flow):
    ms = [MESHES[n]() for n in ("part2", "rows", "hybrid")]
    b = usg.BatchSolver(ms, flow=flow, mach=[0.3, 0.4, 0.35], aoa=[0.0, 2.0, 1.0], reynolds=1e4)
    hb = b.lusgs(4, history=True)
    U, dW = b.U, b.field(usg.F_DW)
    for i, m in enumerate(ms):
        s = usg.Solver(m, flow=flow, mach=[0.3, 0.4, 0.35][i], aoa=[0.0, 2.0, 1.0][i], reynolds=1e4)
        h = s.lusgs(4, history=True)
        assert np.array_equal(U[b.case_slice(i)], s.U)
        assert np.array_equal(dW[b.case_slice(i)], s.field(usg.F_DW))
        assert np.array_equal(hb[:, i], h)


def test_blanked_cells_in_level_sweeps():
    """Hole cells keep their state and give no increment to their neighbours,
    in the first levels of either sweep as elsewhere."""
    m = MESHES["rows"]()
    blank = np.ones(m.nc, np.int32)
    blank[[0, 5, m.nc // 2, m.nc // 2 + 1, m.nc - 1]] = 0
    s = usg.Solver(m, flow=usg.EULER, mach=0.3, aoa=2.0)
    s.set_overset(dict(blank=blank, recv=np.zeros(0, np.int32), off=np.zeros(1, np.int32),
                       donor=np.zeros(0, np.int32), w=np.zeros(0)))
    o = O.OracleSolver(O.OracleMesh(m), O.EULER, 0.3, 2.0, 1e6)
    o.set_blank(blank)
    U0 = s.U
    s.lusgs(4)
    for _ in range(4):
        o.lusgs_step()
    assert np.max(np.abs(s.U - o.U)) <= TOL * np.max(np.abs(o.U))
    assert np.array_equal(s.U[blank == 0], U0[blank == 0])
