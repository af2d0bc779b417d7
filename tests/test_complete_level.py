"""Octrees whose root lies off the origin: the places of a complete level's tiles are relative to the root's cube, and
the cycles that visit complete levels in one launch leave the same bits as on the same octree at the origin."""
import os
import subprocess

import numpy as np
import pytest

import cirrus_amg as P
import helpers as H

RECORD = 4 + 1 + 12 + 44880   # a blob's record: level, type, coordinates, tile


def test_places_of_a_complete_level():
    cpp = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
    subprocess.run(["make", "-s", "-C", cpp, "_build/test_complete_level"], check=True)
    r = subprocess.run([os.path.join(cpp, "_build", "test_complete_level")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "complete_level OK" in r.stdout, r.stdout + r.stderr


def _moved(g, root):
    """The same octree, cell types and operator under a root at `root`, and its tiles' indices in g."""
    blob = bytearray(g.dump_blob())
    rec = np.frombuffer(blob, np.uint8, g.N * RECORD, 40 + 4 * g.num_levels).reshape(g.N, RECORD)
    co = rec[:, 5:17].copy().view(np.int32) + (np.array(root) << rec[:, :4].copy().view(np.int32))
    rec[:, 5:17] = co.astype(np.int32).view(np.uint8)
    m = P.HADeviceGrid.load_blob(bytes(blob))
    lv, co, _ = g.tiles()
    at = {(l, *c): t for t, (l, c) in enumerate(zip(lv.tolist(), co.tolist()))}
    lv, co, _ = m.tiles()
    return m, np.array([at[(l, *c)] for l, c in zip(lv.tolist(), (co - (np.array(root) << lv[:, None])).tolist())])


ROOTS = [(1, 0, 0), (-1, 2, 0), (0, -3, 5)]


@pytest.mark.parametrize("root", ROOTS)
def test_moved_octree_is_the_same(root):
    _, g = H.build_pair("uniform2", with_device=False)
    m, of = _moved(g, root)
    assert m.N == g.N and sorted(of) == list(range(g.N))
    for links in ("neighbors", "parents", "children"):
        a, b = getattr(m, links)(), getattr(g, links)()[of]
        assert np.array_equal(np.where(a >= 0, of[np.maximum(a, 0)], -1), b), links


@pytest.mark.gpu
@pytest.mark.parametrize("root", ROOTS)
@pytest.mark.parametrize("case", ["uniform3", "sphere_solid24"])
@pytest.mark.parametrize("solver", ["rbgs", "jacobi", "gmg", "cmg"])
def test_cycles_under_a_root_off_the_origin(solver, case, root):
    print("\nmoved root", solver, case, root, flush=True)
    _, g = H.build_pair(case)
    m, of = _moved(g, root)
    for ch, seed in ((1, 3), (3, 4)):
        fill = H.random_fill(g.N, seed)
        g.set_channel(ch, fill)
        m.set_channel(ch, fill[of])
    if solver in ("gmg", "cmg"):
        cls = P.GMGSolver if solver == "gmg" else P.CMGSolver
        make, o = lambda grid: cls(grid, 0.5, 0.75), P.default_opts(level_iters=2, coarsest_iters=10)
    else:
        make = lambda grid: P.AMGSolver(grid, H.C0, H.R_MATRIX, 1.0, 1.0)
        jacobi = solver == "jacobi"
        o = P.default_opts(smoother=int(jacobi), mu=2, omega=2.0 / 3.0 if jacobi else 1.5, level_iters=2, coarsest_iters=6)
    for grid in (g, m):
        make(grid).cycle(o, 4, 1, 3)
    for ch in (4, 1, 3):
        a, b = g.channel(ch)[of], m.channel(ch)
        assert np.array_equal(H.bits(a), H.bits(b)), (ch, np.abs(a - b).max())
