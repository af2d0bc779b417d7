"""The quotients of the fused visits (a product with an FP64 reciprocal) against the per-pass kernels' division, bit for
bit, through cycles on an operator without face coefficients, where a pass is b / d alone: all exponents, quotients next
to midpoints, subnormal diagonals, right-hand sides and quotients, zeros, infinities and NaN."""
import numpy as np
import pytest

import cirrus_amg as P
import helpers as H

pytestmark = pytest.mark.gpu
C0 = H.C0


def _pairs(kind, n, rng):
    """n right-hand sides and diagonals (float32)"""
    d = np.ldexp(rng.uniform(1, 2, n), rng.integers(-40, 41, n)).astype(np.float32)
    if kind == "subnormal":
        return (d.astype(np.float64) * rng.uniform(-1, 1, n) * 2.0**-126).astype(np.float32), d
    if kind == "midpoints":
        # a quotient of 25 bits times d, rounded: next to the midpoint of two neighbours
        q = np.ldexp(2.0 * rng.integers(2**23, 2**24, n) + 1, rng.integers(-80, 40, n)) * rng.choice([-1, 1], n)
        return (q * d.astype(np.float64)).astype(np.float32), d
    if kind == "extremes":
        bits = rng.integers(0, 2**32, (2, n), dtype=np.uint64).astype(np.uint32)
        edge = np.array([0, 1, 2, 0x7ffffe, 0x7fffff, 0x400000, 0x3fffff], np.uint32)
        bits = np.where((bits >> 23) & 0xff == 0xff, bits ^ np.uint32(1 << 23), bits)   # finite
        bits = (bits & np.uint32(0xff800000)) | edge[rng.integers(0, 7, (2, n))]
        return bits[0].view(np.float32), bits[1].view(np.float32)
    special = np.array([0, -0.0, np.inf, -np.inf, np.nan, 2.0**-149, 2.0**-126, 3.4e38, 1, -1], np.float32)
    return rng.choice(special, n), rng.choice(special, n)


def _no_ties(n, d):
    """1 in the place of a right-hand side whose quotient lies halfway between two subnormal numbers (the one case in
    which the two may round differently)"""
    with np.errstate(all="ignore"):
        q = np.ldexp(np.abs(n.astype(np.float64) / d.astype(np.float64)), 150)
        return np.where((q < 2.0**24) & (q % 2 == 1), np.float32(1), n)


@pytest.mark.parametrize("level", [2, 1, 0])
@pytest.mark.parametrize("smoother", [0, 1])
@pytest.mark.parametrize("kind", ["subnormal", "midpoints", "extremes", "special"])
def test_quotients_of_fused_visits(kind, smoother, level):
    print("\nquotient", kind, smoother, level, flush=True)
    _, g = H.build_pair("uniform2")
    lv = g.tiles()[0]
    rng = np.random.default_rng(level)
    # above `level` a right-hand side goes down as it is: the cells are DIRICHLET or, on the way to level 0,
    # without diagonal and smoothing; one cell of each block of k^3 cells that becomes one of `level`'s
    types = np.where((lv > level) & (level > 0), P.DIRICHLET, P.INTERIOR).astype(np.uint8)
    g.set_cell_types(np.repeat(types[:, None], 512, 1))
    v = np.arange(512)
    k = 2 ** (2 - level)
    corner = ((v >> 6) % k == 0) & ((v >> 3) % 8 % k == 0) & (v % 8 % k == 0)
    b, d = _pairs(kind, g.N * 512, rng)
    b, d = _no_ties(b, d).reshape(-1, 512), d.reshape(-1, 512)
    if level == 2:
        corner = v % 4 < 3   # some cells with no right-hand side
    rhs = np.where((lv == 2)[:, None] & corner, b, np.float32(0))
    diag = np.where((lv == level)[:, None], d, np.float32(level > 0))
    for a in range(3):
        g.fill_channel(C0 + a, 0.0)
    g.set_channel(C0 + 3, diag)
    out = []
    saved = P.get_kernel_forms()
    for mask in (0, 16):
        g.set_channel(1, rhs)
        g.fill_channel(3, 0.0)
        g.fill_channel(4, 0.0)
        o = P.default_opts(smoother=smoother, mu=1, omega=1.0, level_iters=int(level > 0), coarsest_iters=2)
        try:
            P.set_kernel_forms(mask, 0)
            P.AMGSolver(g, C0, H.R_MATRIX, 1.0, 1.0).cycle(o, 4, 1, 3)
        finally:
            P.set_kernel_forms(saved[0], 0)
        out.append([g.channel(c) for c in (4, 1, 3)])
    for c, x, y in zip((4, 1, 3), *out):
        same = (H.bits(x) == H.bits(y)) | (np.isnan(x) & np.isnan(y))
        assert same.all(), (c, int((~same).sum()), x[~same][:4], y[~same][:4])
    assert np.any(out[0][0][lv == level])
