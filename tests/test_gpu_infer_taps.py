"""Each tap of each layer of the inference kernel alone: a net with one weight of 1 a layer moves the rounded
input, so the result is known to the bit on every cell, at the edges of the volume too."""
import numpy as np
import pytest

import cirrus_amg as P
import helpers as H

pytestmark = pytest.mark.gpu


def _bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


def _moved(v, tap):
    """out[p] = v[p + offset of the tap], 0 outside the volume"""
    p = np.pad(v, ((0, 0), (1, 1), (1, 1), (1, 1)))
    a, b, c = tap // 9, tap // 3 % 3, tap % 3
    return p[:, a:a + 10, b:b + 10, c:c + 10]


@pytest.mark.parametrize("layer", [1, 2, 3])
@pytest.mark.parametrize("case", ["sphere_empty24", "c3_small"])
def test_single_taps(case, layer):
    go, gp = H.build_pair(case)
    go.rhs_uniform(1, 5, True)
    gp.set_channel(1, go.channel(1))
    lv, co, ty = go.tiles()
    T = go.cell_types().reshape(-1, 8, 8, 8)
    leaf = np.where((lv == go.max_level) & (ty == 1))[0]
    d = gp.channel(H.C0 + 3).reshape(-1, 8, 8, 8)
    r = gp.channel(1).reshape(-1, 8, 8, 8)
    x8 = np.where((T == 2) & (d != 0), r / np.where(d != 0, d, 1), 0).astype(np.float32)
    at = {tuple(co[t]): t for t in leaf}
    x = np.zeros((len(leaf), 10, 10, 10), np.float32)
    for n, t in enumerate(leaf):
        x[n, 1:9, 1:9, 1:9] = x8[t]
        for axis in range(3):
            for side in (-1, 1):
                c = list(co[t])
                c[axis] += side
                m = at.get(tuple(c))
                if m is None:
                    continue
                to, of = [slice(1, 9)] * 3, [slice(0, 8)] * 3
                to[axis], of[axis] = (0, 7) if side < 0 else (9, 0)
                x[(n, *to)] = x8[(m, *of)]
    x = _bf16(x)
    solver = P.AMGSolver(gp, H.C0, H.R_MATRIX, 1.0, 1.0)
    rng = np.random.default_rng(layer)
    for tap in range(27):
        taps, c1, c2 = [13, 13, 13], rng.integers(16), rng.integers(16)
        taps[layer - 1] = tap
        w = np.zeros(P.NET_WEIGHTS, np.float32)
        w[c1 * 27 + taps[0]] = 1
        w[432 + (c2 * 16 + c1) * 27 + taps[1]] = 1
        w[7344 + c2 * 27 + taps[2]] = 1
        solver.set_net(w)
        solver.net_infer(1, H.C0 + 3, 6)
        want = x
        for k in range(3):
            want = _moved(want, taps[k])
            want = np.maximum(want, 0) if k < 2 else want
        want = np.where(T[leaf] == 2, want[:, 1:9, 1:9, 1:9], 0)
        got = gp.channel(6).reshape(-1, 8, 8, 8)[leaf]
        assert np.array_equal(got, want), (tap, int((got != want).sum()), len(leaf))
