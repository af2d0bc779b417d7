"""A cycle's visits to complete levels (all of a tile's passes in one launch, its halo computed again), against the
oracle bit for bit: coded and FP32 coefficients, levels with LEAF and NONLEAF tiles, a complete finest level, the
prolongation into a graded level, and the iteration counts up to and beyond what one launch holds."""
import numpy as np
import pytest

import cirrus_amg as P
import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask", [0, 64])
@pytest.mark.parametrize("case", ["uniform2", "uniform3", "c3_small", "sphere_solid24"])
@pytest.mark.parametrize("smoother,mu,level_iters", [(0, 2, 2), (0, 1, 1), (0, 1, 3), (1, 1, 1), (1, 2, 2), (1, 1, 3),
                                                     (1, 1, 4), (1, 1, 5)])
def test_complete_levels_bitexact(case, smoother, mu, level_iters, mask):
    print("\ndense", case, smoother, mu, level_iters, mask, flush=True)
    go, gp = H.build_pair(case)
    omega = 2.0 / 3.0 if smoother else 1.5
    for ch, seed in ((1, 3), (3, 4)):
        fill = H.random_fill(go.N, seed)
        go.channel(ch)[:] = fill
        gp.set_channel(ch, fill)
    o = P.default_opts(smoother=smoother, mu=mu, omega=omega, level_iters=level_iters, coarsest_iters=6)
    c = O.make_cycle(mu=mu, smoother=smoother, omega=omega, level_iters=level_iters, coarsest_iters=6)
    go.fas_cycle(c, 4, 1, 3, H.C0)
    saved = P.get_kernel_forms()
    try:
        P.set_kernel_forms(mask, 0)
        P.AMGSolver(gp, H.C0, H.R_MATRIX, 1.0, 1.0).cycle(o, 4, 1, 3)
    finally:
        P.set_kernel_forms(saved[0], 0)
    for ch in (4, 1, 3):
        a, b = go.channel(ch), gp.channel(ch)
        assert np.array_equal(H.bits(a), H.bits(b)), (ch, np.abs(a - b).max())
