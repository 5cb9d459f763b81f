"""Objects that need more LDS than one made after them still run, with the
same results: the most that a kernel may take belongs to the kernel."""
import numpy as np
import pytest

from tmp_amd import mesh as MM
from tmp_amd import mlp, usg

pytestmark = pytest.mark.gpu


def test_wide_levels_after_a_mesh_of_narrower_ones():
    wide = MM.rect(512, 515, bottom=MM.WALL)
    U = []
    for between in (False, True):
        with usg.Solver(wide, flow=usg.SST, mach=0.3, aoa=2.0, reynolds=1e4) as s:
            if between:
                usg.Solver(MM.rect(20, 40, bottom=MM.WALL), flow=usg.SST, mach=0.3).close()
            s.lusgs(2)
            U.append(s.U)
    assert np.array_equal(U[0], U[1])


def test_deep_network_after_a_shallow_one():
    rng = np.random.default_rng(2)
    x, y = rng.normal(size=(70, 128)).astype(np.float32), rng.normal(size=(70, 4)).astype(np.float32)
    got = []
    for between in (False, True):
        g = mlp.MLP(128, 256, 8, 4)
        g.set_params(*[np.random.default_rng(3).normal(0, 0.1, n) for n in (g.nw, g.nb)])
        if between:
            mlp.MLP(20, 256, 2, 2).close()
        got.append((g.predict(x),) + g.gradients(x, y))
        g.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
