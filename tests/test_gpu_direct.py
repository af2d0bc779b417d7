"""The FP64 direct solve of level 0: its inverse is made on the device for symmetric positive definite systems (sizes off
the elimination's blocks and the largest one among them) and on the host otherwise; both solve the level-0 system.  The
unpivoted elimination inverts an unsymmetric system with positive pivots as well, so no case tells which of the two ran."""
import os
import subprocess

import numpy as np
import pytest

import cirrus_amg as P
import helpers as H

pytestmark = pytest.mark.gpu


def _grid(case):
    """a single-level grid of one tile, or of eight (so that a cycle is the direct solve), its types and operator"""
    g = P.HADeviceGrid(log2_hash=(4,))
    for o in range(8 if case == "largest" else 1):
        g.setTileHost(0, (o & 1, o >> 1 & 1, o >> 2 & 1), P.LEAF)
    g.rebuild()
    g.finalize()
    rng = np.random.default_rng(5)
    types = np.full((g.N, 512), P.INTERIOR, np.uint8)
    if case == "ragged":       # 512 - 75 unknowns: not a multiple of 32
        types[0, rng.choice(512, 75, replace=False)] = P.DIRICHLET
    if case == "few":          # a few unknowns only
        types[:] = P.DIRICHLET
        types[0, rng.choice(512, 20, replace=False)] = P.INTERIOR
    g.set_cell_types(types)
    g.prepare_types_and_coeffs(H.C0, H.R_MATRIX)
    return g


def _matrix(g):
    """the level-0 system from the grid's types and coefficients (a cell without diagonal has an empty row)"""
    C = [g.channel(H.C0 + a).astype(np.float64) for a in range(4)]
    co = g.tiles()[1]
    v = np.arange(512)
    at = (co[:, None] * 8 + np.stack([v >> 6, (v >> 3) & 7, v & 7], 1)).reshape(-1, 3)
    cells = np.where(g.cell_types().ravel() == P.INTERIOR)[0]
    place = {tuple(at[c]): c for c in range(len(at))}
    uid = {c: i for i, c in enumerate(cells)}
    A = np.zeros((len(cells), len(cells)))
    for i, c in enumerate(cells):
        A[i, i] = C[3].ravel()[c]
        if A[i, i] == 0:
            continue
        for a in range(3):
            for side in (-1, 1):
                n = list(at[c])
                n[a] += side
                n = place.get(tuple(n))
                if n in uid:
                    A[i, uid[n]] += C[a].ravel()[c if side < 0 else n]
    return cells, A


@pytest.mark.parametrize("case", ["full", "ragged", "few", "largest", "indefinite", "singular", "unsymmetric"])
def test_level0_direct_solve(case):
    print("\ndirect", case, flush=True)
    g = _grid(case)
    if case in ("indefinite", "singular", "unsymmetric"):
        # a diagonal of its own for one cell: not definite where it is negative; 0 leaves the cell's row empty
        # and the system singular, and with the shift of a pure Neumann system regular and unsymmetric
        d = g.channel(H.C0 + 3)
        d[0, 77] = -8.0 if case == "indefinite" else 0.0
        g.set_channel(H.C0 + 3, d)
    cells, A = _matrix(g)
    b = H.random_fill(g.N, 9)
    g.set_channel(1, b)
    o = P.default_opts(cycle=P.CYCLE_FAS_V, smoother=P.SMOOTH_JACOBI, coarsest_direct=1,
                       is_pure_neumann=int(case == "unsymmetric"))
    if case == "unsymmetric":
        assert not np.array_equal(A, A.T)
        A = A + np.trace(A) / len(cells) ** 2
    s = P.AMGSolver(g, H.C0, H.R_MATRIX, 1.0, 1.0)
    if case == "singular":
        with pytest.raises(P.CmgError) as e:
            s.cycle(o, 4, 1, 3)
        assert "singular" in str(e.value)
        return
    s.cycle(o, 4, 1, 3)
    x = np.linalg.solve(A, b.ravel()[cells].astype(np.float64))
    z = g.channel(4).ravel()
    # the FP32 result of an FP64 solve: half an ulp, and the FP64 error of a condition number below 1e4
    assert np.abs(z[cells] - x).max() <= 2.0**-24 * np.abs(x).max() * 1.01
    rest = np.setdiff1d(np.arange(z.size), cells)
    assert not z[rest].any()


def test_pure_neumann_solve():
    """an all-Neumann box: the level-0 system is the singular one with its constant part shifted"""
    _, gp = H.build_pair("uniform2")
    co = gp.tiles()[1]
    types = gp.cell_types()
    v = np.arange(512)
    for t in np.where(gp.tiles()[2] == 1)[0]:
        at = co[t] * 8 + np.stack([v >> 6, (v >> 3) & 7, v & 7], 1)
        types[t, ((at == 0) | (at == 31)).any(1)] = P.NEUMANN
    gp.set_cell_types(types)
    gp.prepare_types_and_coeffs(H.C0, H.R_MATRIX)
    gp.rhs_uniform(1, 3, True)
    o = P.default_opts(cycle=P.CYCLE_FAS_V, smoother=P.SMOOTH_JACOBI, omega=2.0 / 3.0, coarsest_direct=1)
    it, rel = P.AMGSolver(gp, H.C0, H.R_MATRIX, 1.0, 1.0).solve(relative_tolerance=1e-6, is_pure_neumann=True, opts=o)
    assert rel < 1e-6 and it < 40


def test_no_room_for_the_device_inverse():
    """the workspace's allocation refused (from the host, by the test program's own hipMalloc): the same solution"""
    cpp = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
    subprocess.run(["make", "-s", "-C", cpp, "_build/test_inverse_fallback"], check=True)
    print("\ninverse fallback", flush=True)
    r = subprocess.run([os.path.join(cpp, "_build", "test_inverse_fallback")], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "inverse fallback OK" in r.stdout, r.stdout + r.stderr
