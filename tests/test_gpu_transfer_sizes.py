"""Fields read back at sizes on both sides of the change between a launch into
the pinned buffers and the runtime's copy into them (16 KB; 10 000 FP64 values,
50 000 FP32 values): what was set comes back bit for bit."""
import numpy as np
import pytest

from tmp_amd import mesh as MM
from tmp_amd import usg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj", [(16, 32), (27, 19), (32, 64), (3, 683), (50, 50), (41, 61), (50, 100), (100, 100), (73, 137)])
def test_fields_of_one_to_four_values(ni, nj):
    m = MM.rect(ni, nj, bottom=MM.WALL)
    r = np.random.default_rng(ni)
    U, W = r.uniform(1, 2, (ni * nj, 4)), r.uniform(1, 2, (ni * nj, 4))
    T, TW, mut = r.uniform(1, 2, (ni * nj, 2)), r.uniform(1, 2, (ni * nj, 2)), r.uniform(1, 2, ni * nj)
    with usg.Solver(m, flow=usg.SST) as s:
        s.set_state(U, W, T, TW, mut)
        for fid, want in ((usg.F_PRIM, U), (usg.F_CONS, W), (usg.F_TURB, T), (usg.F_TCONS, TW), (usg.F_MUT, mut)):
            assert np.array_equal(s.field(fid), want)


@pytest.mark.parametrize("ni,nj", [(16, 32), (27, 19), (50, 125), (7, 893), (250, 200), (77, 650)])
def test_fp32_fields(ni, nj):
    """FP32 gradients of a state linear in y, each variable with its own slope:
    exact but for the roundings of an interior cell's sum (under 50 of 2^-24 of
    the largest slope)."""
    m = MM.rect(ni, nj, lx=1.0, ly=1.0)
    y = (np.arange(ni * nj) % nj + 0.5) / nj
    U = np.stack([1 + 0.1 * y, 1 / 1.4 + 0.2 * y, 0.3 * y, 0.4 * y], 1)
    with usg.Solver(m, flow=usg.LAMINAR, mach=0.5, reynolds=5000.0, precision=usg.MIXED) as s:
        s.set_prim(U)
        s.residual()
        g = s.field(usg.F_GRAD).reshape(ni, nj, 4, 2)[1:-1, 1:-1]
        bar = 50 * 2.0 ** -24 * 0.4
        assert np.max(np.abs(g[..., 0])) <= bar
        assert np.max(np.abs(g[..., 1] - np.array([0.1, 0.2, 0.3, 0.4]))) <= bar
