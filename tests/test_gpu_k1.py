"""BSE_K1! from the sums over the K2 boxes and of Π, and the weight sums that BSE_K2! takes (k_k1, k_bse_w), against
the oracle: boxes smaller and larger than the reference vertex's, a bubble mesh narrower than the K2 boxes, one
narrower than the reference vertex's, more than one wavefront of terms, a channel alone and all three, with and
without groups.  The sums hold the oracle's products, a few hundred of order one, in another order: 1e-12 is over
ten times their rounding."""
import pytest

import pyoracle as po
from helpers import BOX, make_pair, relerr

pytestmark = pytest.mark.gpu
TOL = 1e-12
BOXES = {
    "smallest": dict(BOX, nG=4, nK1=1, nK2=(1, 1), nK3=(1, 1), mPinu=1),
    "small": dict(BOX, nG=8, nK1=4, nK2=(2, 3), nK3=(1, 2), mPinu=4),
    "large": dict(BOX, nG=12, nK1=12, nK2=(9, 11), nK3=(2, 2), mPinu=1),
    "wide": dict(BOX, nG=20, nK1=36, nK2=(2, 35), nK3=(1, 2), mPinu=2),
}


@pytest.mark.parametrize("groups", [False, True])
@pytest.mark.parametrize("box", list(BOXES))
@pytest.mark.parametrize("case", ["local_ref", "local_vertexref", "nl_L2", "nl_L3"])
def test_k1(case, box, groups):
    import fdga
    from fdga import _lib as ids
    S, O = make_pair(case, seed=13, box=BOXES[box])
    if groups:
        S.init_sym_grp()
        O.init_sym_grp()
    for ch in (po.PCH, po.ACH, po.TCH):
        fdga.BSE_L_K2(S, ch)
        O.bse_l_k2(ch)
    for ch in (po.PCH, po.ACH, po.TCH):
        fdga.BSE_K1(S, ch)
        O.bse_k1(ch)
    for ch in (po.PCH, po.ACH, po.TCH):
        fdga.BSE_K2(S, ch)
        O.bse_k2(ch)
    for ch in range(3):
        for cls in (1, 2):
            e = relerr(S.get(ids.vertex_id(1, ch, cls)), O.get(po.vertex_id(po.VTX_FBUFF, ch, cls)))
            assert e < TOL, f"K{cls} channel {ch}: {e:.3e}"
    for strategy, st in (("fdPA", po.FDPA), ("scPA", po.SCPA)):
        fdga.iterate_solver(S, strategy)
        O.iterate(st)
        assert relerr(fdga.flatten(S), O.flatten()) < TOL
