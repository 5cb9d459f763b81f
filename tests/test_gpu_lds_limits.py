"""Objects that need more LDS than one made after them still run, with the
same results: the most that a kernel may take belongs to the kernel."""
import numpy as np
import pytest

from tmp_amd import mesh as MM
from tmp_amd import usg

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
