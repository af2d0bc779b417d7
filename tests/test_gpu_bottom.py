"""The bottom two levels of a FAS cycle in one workgroup, against the oracle bit for bit, over the sweep counts,
smoothers and repetitions that change its path; and the formula of the quotient it divides with (the device's own
reciprocal: test_gpu_quotient.py)."""
import numpy as np
import pytest

import cirrus_amg as P
import helpers as H
import oracle as O


def test_quotient_through_fp64_reciprocal():
    """float(double(n) * (1 / double(d))) is the correctly rounded n / d: all exponents, random and extreme mantissas"""
    rng = np.random.default_rng(1)
    bits = rng.integers(0, 2**32, (2, 4_000_000), dtype=np.uint64).astype(np.uint32)
    edge = np.array([0, 1, 2, 0x7ffffe, 0x7fffff, 0x400000, 0x3fffff], np.uint32)
    bits[0, :1_000_000] = (bits[0, :1_000_000] & 0xff800000) | edge[rng.integers(0, 7, 1_000_000)]
    bits[1, 500_000:1_500_000] = (bits[1, 500_000:1_500_000] & 0xff800000) | edge[rng.integers(0, 7, 1_000_000)]
    n, d = bits.view(np.float32)
    with np.errstate(all="ignore"):
        want = n / d
        got = (n.astype(np.float64) * (1.0 / d.astype(np.float64))).astype(np.float32)
    normal = ~(np.abs(want) < np.finfo(np.float32).tiny) | (want == 0)   # a subnormal quotient may be a tie
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same[normal].all()
    assert (np.abs(got.astype(np.float64) - want.astype(np.float64))[~normal & np.isfinite(want)] <= 2.0**-149).all()


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["uniform2", "sphere_empty24"])
@pytest.mark.parametrize("smoother,mu,level_iters,coarsest_iters", [
    (0, 2, 2, 10), (0, 1, 1, 1), (0, 3, 1, 2), (0, 2, 3, 0), (0, 1, 0, 6), (0, 2, 1, 7),
    (1, 2, 2, 10), (1, 1, 1, 1), (1, 3, 3, 2), (1, 2, 2, 0), (1, 1, 0, 5)])
def test_bottom_levels_bitexact(case, smoother, mu, level_iters, coarsest_iters):
    print("\nbottom", case, smoother, mu, level_iters, coarsest_iters, flush=True)
    go, gp = H.build_pair(case)
    omega = 2.0 / 3.0 if smoother else 1.5
    for ch, seed in ((1, 3), (3, 4)):
        fill = H.random_fill(go.N, seed)
        go.channel(ch)[:] = fill
        gp.set_channel(ch, fill)
    o = P.default_opts(smoother=smoother, mu=mu, omega=omega, level_iters=level_iters, coarsest_iters=coarsest_iters)
    c = O.make_cycle(mu=mu, smoother=smoother, omega=omega, level_iters=level_iters, coarsest_iters=coarsest_iters)
    go.fas_cycle(c, 4, 1, 3, H.C0)
    P.AMGSolver(gp, H.C0, H.R_MATRIX, 1.0, 1.0).cycle(o, 4, 1, 3)
    # z, and the right-hand sides and saved x that the cycle leaves on the coarse levels
    for ch in (4, 1, 3):
        a, b = go.channel(ch), gp.channel(ch)
        assert np.array_equal(H.bits(a), H.bits(b)), (ch, np.abs(a - b).max())
