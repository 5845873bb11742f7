"""The far terms of the is_mfRG and _new forms of BSE_K1! and BSE_K2! (far_terms) against the oracle: no far part (the
window covers the mesh), a band that ends at the mesh, more far entries than lanes, with and without groups.  The sums
hold the oracle's products, a few hundred of order one, in another order: 1e-12 is over ten times their rounding."""
import numpy as np
import pytest

import pyoracle as po
from helpers import BOX, make_pair

pytestmark = pytest.mark.gpu
TOL = 1e-12
BOXES = {
    "no far part": dict(BOX, nG=6, nK1=3, nK2=(2, 2), nK3=(1, 1), mPinu=1),
    "to the end of the mesh": dict(BOX, nG=16, nK1=20, nK2=(3, 4), nK3=(2, 2), mPinu=2),
    "beyond the band": dict(BOX, nG=8, nK1=5, nK2=(4, 5), nK3=(2, 2), mPinu=12),
    "more than a wave": dict(BOX, nG=20, nK1=50, nK2=(2, 40), nK3=(1, 2), mPinu=3),
}


@pytest.mark.parametrize("groups", [False, True])
@pytest.mark.parametrize("box", list(BOXES))
@pytest.mark.parametrize("case", ["local_ref", "local_vertexref", "nl_L2"])
def test_forms(case, box, groups):
    import fdga
    S, O = make_pair(case, seed=17, box=BOXES[box])
    rng = np.random.default_rng(18)
    for ch in range(3):
        for cls in (1, 2):
            v = 0.2 * (rng.standard_normal(S.vertex(2, ch, cls).size) + 1j * rng.standard_normal(S.vertex(2, ch, cls).size))
            S.set_vertex(2, ch, cls, v)
            O.set_vertex(po.VTX_FL, ch, cls, v)
    if groups:
        S.init_sym_grp()
        O.init_sym_grp()
    for name, cls, dev, orc, mfrg in (("K1 mfRG", 1, fdga.BSE_K1, O.bse_k1, True), ("K2 mfRG", 2, fdga.BSE_K2, O.bse_k2, True),
                                      ("K1_new", 1, fdga.BSE_K1_new, O.bse_k1_new, False),
                                      ("K2_new", 2, fdga.BSE_K2_new, O.bse_k2_new, False)):
        for ch in (po.PCH, po.ACH, po.TCH):
            dev(S, ch, mfrg)
            orc(ch, mfrg)
        for ch in range(3):
            a, b = S.vertex(1, ch, cls), O.vertex(po.VTX_FBUFF, ch, cls)
            s = np.max(np.abs(b))
            e = np.max(np.abs(a - b)) / (s if s > 0 else 1.0)   # (the local mfRG K1 has a zero t channel)
            assert e < TOL, (name, ch, e)
    S.close()
