"""Several threads on one context: fields of several transfer buffers read side
by side give what a single thread reads, bit for bit."""
import threading

import numpy as np
import pytest

from tmp_amd import mesh as MM
from tmp_amd import usg

pytestmark = pytest.mark.gpu


def test_fields_read_side_by_side():
    m = MM.rect(300, 301, bottom=MM.WALL)
    with usg.Solver(m, flow=usg.LAMINAR, mach=0.5, aoa=2.0, reynolds=5000.0) as s:
        s.set_prim(np.array([1.0, 1.0 / 1.4, 0.3, 0.1]) + 0.01 * np.random.default_rng(1).uniform(-1, 1, (s.nc, 4)))
        s.residual()
        want = {f: s.field(f) for f in (usg.F_PRIM, usg.F_GRAD, usg.F_LAMC)}
        forces, bad = s.forces(), []

        def fields(f):
            bad.extend(f for _ in range(20) if not np.array_equal(s.field(f), want[f]))

        def values():
            bad.extend("forces" for _ in range(100) if s.forces() != forces)

        ts = [threading.Thread(target=fields, args=(f,)) for f in want] + [threading.Thread(target=values)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not bad, bad
