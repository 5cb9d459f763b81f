"""Work lists of 64-item chunks: the gradient kernel at cell counts around a
chunk and around eight parts of one, against the oracle; the face kernel on
both sides of the size from which it takes chunks, against the fused
face-cell launch, whose tiles come from another list."""
import numpy as np
import pytest

from oracle import oracle as O
from tmp_amd import mesh as MM
from tmp_amd import usg

pytestmark = pytest.mark.gpu


def _state(nc, seed):
    r = np.random.default_rng(seed)
    return np.array([1.0, 1.0 / 1.4, 0.3, 0.1]) + 0.01 * r.uniform(-1, 1, (nc, 4))


@pytest.mark.parametrize("ni,nj", [(1, 1), (9, 7), (8, 8), (13, 5), (73, 7), (64, 8), (57, 9)])
@pytest.mark.parametrize("renumbered", [False, True])
def test_gradient_chunks(ni, nj, renumbered):
    m = MM.rect(ni, nj, jitter=0.1, seed=3, bottom=MM.WALL)
    if renumbered:
        m = usg.mesh_renumber(m)[0]
    U = _state(ni * nj, 1)
    orc = O.OracleSolver(O.OracleMesh(m), O.LAMINAR, 0.5, 2.0, 5000.0)
    orc.set_prim(U)
    orc.residual()
    with usg.Solver(m, flow=usg.LAMINAR, mach=0.5, aoa=2.0, reynolds=5000.0) as s:
        s.set_prim(U)
        s.residual()
        # the parity bar of one residual: libm's last bits at far-field faces
        for got, want in ((s.field(usg.F_GRAD), orc.field("gradU", 8)), (s.field(usg.F_PHI), orc.field("phi", 4)),
                          (s.R, orc.R)):
            want = np.asarray(want).reshape(got.shape)
            assert np.max(np.abs(got - want)) <= 1e-13 * np.max(np.abs(want))


@pytest.mark.parametrize("ni,nj", [(500, 500), (501, 499), (641, 390)])
def test_face_chunks(ni, nj):
    """250 000 Euler cells are the last that take indices."""
    m = usg.mesh_renumber(MM.rect(ni, nj, bottom=MM.WALL))[0]
    U = _state(ni * nj, 2)
    R = []
    for fused in (False, True):
        with usg.Solver(m, flow=usg.EULER, mach=0.5, aoa=2.0) as s:
            s.fused(fused)
            s.set_prim(U)
            s.residual()
            R.append(s.R)
    assert np.array_equal(R[0], R[1])
