"""The local solver's BSE_L_K2!, BSE_K2! and SDE L-vertices as sums over the classes' intervals (k_seg_k2,
k_seg_sde) against the oracle, where an interval can go wrong: the smallest boxes, boxes larger and smaller
than the reference vertex's, a bubble mesh narrower than the boxes (every interval cut at its ends), more than
one wavefront of terms per class, a channel alone and the three together.  The sums hold the same products as
the oracle's in another order, a few hundred terms of order one: 1e-12 is some 30 times their rounding."""
import pytest

import pyoracle as po
from helpers import BOX, make_pair, relerr

pytestmark = pytest.mark.gpu
TOL = 1e-12
BOXES = {
    "smallest": dict(BOX, nG=4, nK1=1, nK2=(1, 1), nK3=(1, 1), mPinu=1),
    "unequal": dict(BOX, nG=12, nK1=9, nK2=(7, 3), nK3=(2, 3), mPinu=1),
    "narrow mesh": dict(BOX, nG=12, nK1=8, nK2=(8, 8), nK3=(5, 4), mPinu=1),
    "wide": dict(BOX, nG=60, nK1=40, nK2=(9, 34), nK3=(6, 33), mPinu=3),
}


def _check(S, O, vtx, ovtx, what):
    from fdga import _lib as ids
    for ch in range(3):
        e = relerr(S.get(ids.vertex_id(vtx, ch, 2)), O.get(po.vertex_id(ovtx, ch, 2)))
        assert e < TOL, f"{what} channel {ch}: {e:.3e}"


@pytest.mark.parametrize("groups", [False, True])
@pytest.mark.parametrize("box", list(BOXES))
@pytest.mark.parametrize("case", ["local_ref", "local_vertexref"])
def test_intervals(case, box, groups):
    import fdga
    from fdga import _lib as ids
    S, O = make_pair(case, seed=7, box=BOXES[box])
    if groups:
        S.init_sym_grp()
        O.init_sym_grp()
    for ch in (po.PCH, po.ACH, po.TCH):
        fdga.BSE_L_K2(S, ch)
        O.bse_l_k2(ch)
    _check(S, O, 2, po.VTX_FL, "L_K2")
    for ch in (po.PCH, po.ACH, po.TCH):
        fdga.BSE_K2(S, ch)
        O.bse_k2(ch)
    _check(S, O, 1, po.VTX_FBUFF, "K2")
    fdga.SDE(S, "fdPA")
    O.sde(po.FDPA)
    assert relerr(S.get(ids.SIGMA), O.get(po.SIGMA)) < TOL
    fdga.iterate_solver(S, "fdPA")
    O.iterate(po.FDPA)
    _check(S, O, 2, po.VTX_FL, "iterate L_K2")
    assert relerr(fdga.flatten(S), O.flatten()) < TOL
