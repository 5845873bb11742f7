"""The local solver's BSE_L_K2! of one channel on both sides of the line between its two forms, point by point up to two
million sums and as segments of prepared weights beyond, against the oracle; with groups the first form serves both
boxes, over the classes.  Each sum holds the oracle's some hundred products of order one in another order: 1e-12 is over
ten times their rounding."""
import pytest

import pyoracle as po
from helpers import BOX, make_pair, relerr

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("groups", [False, True])
@pytest.mark.parametrize("n2", [42, 43])   # 83 x 84 outputs x 294 frequencies = 2.05 M; 85 x 86 x 298 = 2.18 M
@pytest.mark.parametrize("case", ["local_ref", "local_vertexref"])
def test_both_sides(case, n2, groups):
    import fdga
    from fdga import _lib as ids
    S, O = make_pair(case, seed=23, box=dict(BOX, nG=64, nK1=60, nK2=(n2, n2), nK3=(2, 3), mPinu=6))
    if groups:
        S.init_sym_grp()
        O.init_sym_grp()
    for ch in (po.PCH, po.ACH, po.TCH):
        fdga.BSE_L_K2(S, ch)
        O.bse_l_k2(ch)
    for ch in range(3):
        e = relerr(S.get(ids.vertex_id(2, ch, 2)), O.get(po.vertex_id(po.VTX_FL, ch, 2)))
        assert e < TOL, (ch, e)
    S.close()
