"""Fields to and from the host at sizes around a transfer buffer (65536 values:
16384 cells of four) and past all four buffers: what set_prim and set_state put
in comes back bit for bit, and the derived conserved variables agree."""
import numpy as np
import pytest

from oracle import oracle as O
from tmp_amd import mesh as MM
from tmp_amd import usg

pytestmark = pytest.mark.gpu

SHAPES = [(3, 2), (127, 129), (128, 128), (145, 113), (256, 256), (300, 301)]


def _prim(nc, seed):
    r = np.random.default_rng(seed)
    U = r.uniform(-0.5, 0.5, (nc, 4))
    U[:, :2] += 1.5  # density and pressure
    return U


@pytest.mark.parametrize("ni,nj", SHAPES)
def test_fields_come_back(ni, nj):
    m = MM.rect(ni, nj, bottom=MM.WALL)
    with usg.Solver(m, flow=usg.SST) as s:
        nc = s.nc
        for seed in (1, 2):  # the second through used buffers
            U, T = _prim(nc, seed), _prim(nc, seed + 8)[:, :2].copy()
            s.set_prim(U, T)
            assert np.array_equal(s.U, U)
            assert np.array_equal(s.field(usg.F_TURB), T)
            # one multiplication each
            assert np.array_equal(s.field(usg.F_TCONS), T * U[:, :1])
        W, TW = _prim(nc, 3), _prim(nc, 4)[:, :2].copy()
        mut = _prim(nc, 5)[:, 0].copy()
        s.set_state(U, W, T, TW, mut)
        for fid, want in ((usg.F_PRIM, U), (usg.F_CONS, W), (usg.F_TURB, T), (usg.F_TCONS, TW), (usg.F_MUT, mut)):
            assert np.array_equal(s.field(fid), want)


def test_wide_and_single_fields():
    """Widths 8, 4, 2 and 1 over several buffers: against the oracle at the
    parity bar of a single residual (1e-13), and FP32 arrays of the mixed mode
    against those at its bar (1e-4 of the largest value)."""
    m = MM.rect(150, 111, bottom=MM.WALL)
    U = _prim(150 * 111, 6) * 0.01 + np.array([1.0, 1.0 / 1.4, 0.3, 0.0])
    orc = O.OracleSolver(O.OracleMesh(m), O.LAMINAR, 0.5, 2.0, 5000.0)
    orc.set_prim(U)
    orc.residual()
    want = {usg.F_RES: orc.R, usg.F_GRAD: orc.field("gradU", 8), usg.F_PHI: orc.field("phi", 4),
            usg.F_GRADT: orc.field("gradT", 2), usg.F_LAMC: orc.field("lamc", 1)}
    for precision, bar in ((usg.FP64, 1e-13), (usg.MIXED, 1e-4)):
        with usg.Solver(m, flow=usg.LAMINAR, mach=0.5, aoa=2.0, reynolds=5000.0, precision=precision) as s:
            s.set_prim(U)
            s.residual()
            fields = want if precision == usg.FP64 else (usg.F_GRAD, usg.F_GRADT)
            for f in fields:
                got, ref = s.field(f), np.asarray(want[f]).reshape(s.field(f).shape)
                assert np.max(np.abs(got - ref)) <= bar * np.max(np.abs(ref)), (precision, f)
            l2 = s.res_l2()
            assert np.isfinite(l2) and l2 > 0
