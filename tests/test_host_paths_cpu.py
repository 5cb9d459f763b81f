"""The library's host code over a stand-in HIP runtime (fake_hip.c): what
must hold whatever the kernels compute.  Each case is a program of its own, as
the stand-in has to be loaded before libusg.so."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

HEAD = """
import ctypes, sys, threading
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
from tmp_amd import mesh, usg
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["gcc", "-O2", "-std=gnu11", "-shared", "-fPIC", os.path.join(HERE, "fake_hip.c"), "-o", so],
                   check=True)
    return so


def run(fake, body):
    r = subprocess.run([sys.executable, "-c", HEAD + body, fake, os.path.dirname(HERE)], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_calls_of_several_threads_on_one_context(fake):
    """Fields of several transfer buffers read by one thread beside another
    that reads a second field, and a third that sets the same state again:
    every read gives its own field's values."""
    run(fake, """
m = mesh.rect(300, 301, bottom=mesh.WALL)
s = usg.Solver(m, flow=usg.EULER)
r = np.random.default_rng(1)
U, W = r.uniform(1, 2, (s.nc, 4)), r.uniform(3, 4, (s.nc, 4))
s.set_state(U, W)
bad = []
def read(fid, want):
    for _ in range(40):
        if not np.array_equal(s.field(fid), want):
            bad.append(fid)
def write():
    for _ in range(20):
        s.set_state(U, W)
def small():
    for _ in range(200):
        if s.forces() != (0.0, 0.0):
            bad.append("forces")
ts = [threading.Thread(target=read, args=a) for a in ((usg.F_PRIM, U), (usg.F_CONS, W))]
ts += [threading.Thread(target=write), threading.Thread(target=small)]
for t in ts: t.start()
for t in ts: t.join()
assert not bad, bad
""")


def test_refused_copy_of_the_error_flags_is_an_error(fake):
    """A check of a residual whose flags could not be fetched is not a pass,
    neither the first one nor one after a good one."""
    run(fake, """
import os
for good in (0, 1):
    s = usg.Solver(mesh.rect(4, 3), flow=usg.EULER)
    for _ in range(good):
        s.residual()
    os.environ["FAKE_HIP_REFUSE"] = "k_err_host"
    try:
        s.residual()
    except usg.UsgError as e:
        assert "invalid argument" in str(e), e
    else:
        raise SystemExit("the check passed")
    os.environ["FAKE_HIP_REFUSE"] = ""
    s.residual()
""")


def test_wide_levels_after_a_mesh_of_narrower_ones(fake):
    """The most LDS a kernel may take belongs to the kernel, not to the mesh:
    a solver with a ring of 98 KB still runs when one with 4 KB was made after
    it."""
    run(fake, """
wide = usg.Solver(mesh.rect(512, 515, bottom=mesh.WALL), flow=usg.SST)
narrow = usg.Solver(mesh.rect(20, 40, bottom=mesh.WALL), flow=usg.SST)
for s in (narrow, wide, narrow):
    s.graphs(False)  # the stand-in has none
    s.lusgs(2)
""")


def test_deep_network_after_a_shallow_one(fake):
    """As above for the networks of one width: rows of all layers in LDS."""
    run(fake, """
from tmp_amd import mlp
def use(g):
    g.gradients(np.zeros((5, g.nin)), np.zeros((5, g.nout)))
    g.predict(np.zeros((5, g.nin)))
deep, shallow = mlp.MLP(128, 256, 8, 4), mlp.MLP(20, 256, 2, 2)
for g in (shallow, deep, shallow):
    use(g)
""")


def test_more_layers_than_a_grid_has_rows(fake):
    """A network of more than 65536 layers: its weights are packed layer by
    layer, and a launch has at most 65536 blocks along y."""
    run(fake, """
from tmp_amd import mlp
mlp.MLP(1, 64, 65540, 1).close()
""")


def test_groups_of_the_level_sweeps_meet_the_same_barriers(fake):
    """For levels of one cell to the widest, chunks and rounds around their
    sizes, and batches with cases of no narrow level."""
    run(fake, """
ms = [mesh.rect(a, b, jitter=0.1, seed=1, bottom=mesh.WALL)
      for a, b in ((2, 30), (9, 40), (63, 70), (64, 70), (65, 70), (129, 150), (256, 260), (257, 260), (512, 515), (513, 515))]
ms.append(mesh.airfoil_hybrid(ni=64, dy1=1e-3, rfar=10.0))
one = [usg.Solver(m, flow=usg.EULER) for m in ms]
assert all(sum(s.waves()) > 14 for s in one)
for s in one + [usg.BatchSolver([mesh.rect(1, 1)] + ms[i:] + [mesh.rect(2, 2)], flow=usg.EULER) for i in (0, 3, 7)]:
    s.graphs(False)  # the stand-in has none
    s.lusgs(1)
""")
