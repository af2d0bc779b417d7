"""The geometric V-cycle's complete levels (all of a tile's passes in one launch) and single-tile level 0 (all of its
iterations in one) against the oracle bit for bit, over the iteration counts that change the path, with NEUMANN cells."""
import numpy as np
import pytest

import cirrus_amg as P
import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level_iters,coarsest_iters", [(1, 2), (2, 1), (2, 10), (3, 4), (0, 6)])
@pytest.mark.parametrize("case", ["uniform2", "uniform3", "center_point14", "sphere_solid24", "c2_small"])
@pytest.mark.parametrize("family", [(P.GMGSolver, O.GEO_GMG), (P.CMGSolver, O.GEO_CMG)], ids=["gmg", "cmg"])
def test_geo_vcycle_bitexact(family, case, level_iters, coarsest_iters):
    cls, mode = family
    print("\ngeo dense", case, mode, level_iters, coarsest_iters, flush=True)
    go, gp = H.build_pair(case)
    for ch, seed in ((1, 51), (3, 52), (4, 53)):
        fill = H.random_fill(go.N, seed)
        go.channel(ch)[:] = fill
        gp.set_channel(ch, fill)
    O.lib().og_geo_vcycle(go.h, mode, 4, 1, 3, level_iters, coarsest_iters, np.float32(0.5), np.float32(0.75))
    cls(gp, 0.5, 0.75).cycle(P.default_opts(level_iters=level_iters, coarsest_iters=coarsest_iters), 4, 1, 3)
    for ch in (4, 3):
        a, b = go.channel(ch), gp.channel(ch)
        assert np.array_equal(H.bits(a), H.bits(b)), (ch, np.abs(a - b).max())
