"""The local solver's BSE_L_K2! and BSE_K2! on both sides of the line between their two forms, weights per wave in LDS
with K2 read in place and prepared weights with K2 copied along its diagonals, against the oracle: the largest band of
the first form (128), one below it, and the first of the second (129), with and without groups; a channel alone and
the three together; and the lattice BSE_K2! on its own, whose weights and sums are one launch.  The sums hold the
oracle's products, some hundred of order one, in another order: 1e-12 is over ten times their rounding."""
import pytest

import pyoracle as po
from helpers import BOX, make_pair, relerr

pytestmark = pytest.mark.gpu
TOL = 1e-12
BOXES = {   # band: nK1 + 1 + max(nK1 - 1, n2b - 1 + n2f) + 3
    127: dict(BOX, nG=20, nK1=62, nK2=(4, 5), nK3=(2, 3), mPinu=3),
    128: dict(BOX, nG=20, nK1=62, nK2=(2, 61), nK3=(2, 3), mPinu=3),
    129: dict(BOX, nG=20, nK1=63, nK2=(4, 5), nK3=(3, 5), mPinu=3),
    "129 wide": dict(BOX, nG=20, nK1=63, nK2=(2, 62), nK3=(2, 3), mPinu=3),
}


@pytest.mark.parametrize("groups", [False, True])
@pytest.mark.parametrize("band", list(BOXES))
@pytest.mark.parametrize("case", ["local_ref", "local_vertexref"])
def test_both_sides(case, band, groups):
    import fdga
    from fdga import _lib as ids
    S, O = make_pair(case, seed=19, box=BOXES[band])
    if groups:
        S.init_sym_grp()
        O.init_sym_grp()
    for stage, orc, vtx, ovtx in ((fdga.BSE_L_K2, O.bse_l_k2, 2, po.VTX_FL), (fdga.BSE_K2, O.bse_k2, 1, po.VTX_FBUFF)):
        for ch in (po.PCH, po.ACH, po.TCH):
            stage(S, ch)
            orc(ch)
        for ch in range(3):
            e = relerr(S.get(ids.vertex_id(vtx, ch, 2)), O.get(po.vertex_id(ovtx, ch, 2)))
            assert e < TOL, (stage.__name__, ch, e)
    for strategy, st in (("fdPA", po.FDPA), ("scPA", po.SCPA)):
        fdga.iterate_solver(S, strategy)
        O.iterate(st)
        assert relerr(fdga.flatten(S), O.flatten()) < TOL, strategy
    S.close()


@pytest.mark.parametrize("groups", [False, True])
@pytest.mark.parametrize("nK1,nK2", [(1, (1, 1)), (9, (9, 2)), (40, (3, 6))])
def test_lattice_k2_alone(nK1, nK2, groups):
    import fdga
    from fdga import _lib as ids
    S, O = make_pair("nl_L2", seed=20, box=dict(BOX, nG=12, nK1=nK1, nK2=nK2, nK3=(1, 1), mPinu=2))
    if groups:
        S.init_sym_grp()
        O.init_sym_grp()
    for ch in (po.PCH, po.ACH, po.TCH):
        fdga.BSE_K2(S, ch)
        O.bse_k2(ch)
    for ch in range(3):
        assert relerr(S.get(ids.vertex_id(1, ch, 2)), O.get(po.vertex_id(po.VTX_FBUFF, ch, 2))) < TOL, ch
    S.close()
