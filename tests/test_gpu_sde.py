"""The lattice SDE L-vertices (k_sde_L_nl) where its split of the K3 sums can go wrong: the smallest box, boxes
whose columns leave lanes and column groups idle, a column longer than the block (130 and 260 rows of ν) and more
summed frequencies than are staged at a time (520), a mesh that cuts the sums, one level and two; and K3 held in
FP32 against the same values in FP64.  The sums hold the same products in another order, at most some thousand
terms of order one: 1e-12 is over ten times their rounding."""
import pytest

import pyoracle as po
from helpers import BOX, make_pair, relerr

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("n2b,n3", [(1, (1, 1)), (3, (2, 5)), (4, (3, 33)), (2, (2, 130)), (1, (1, 260))])
@pytest.mark.parametrize("case", ["nl_L2", "nl_L3"])
def test_boxes(case, n2b, n3):
    import fdga
    from fdga import _lib as ids
    box = dict(BOX, nG=6, nK1=max(n3[1], 4), nK2=(n2b, n3[1] + 1 if n3[1] < 4 else n3[1]), nK3=n3, mPinu=1)
    S, O = make_pair(case, seed=11, box=box)
    for strategy, st in (("fdPA", po.FDPA), ("scPA", po.SCPA)):
        fdga.SDE(S, strategy)
        O.sde(st)
        assert relerr(S.get(ids.SIGMA), O.get(po.SIGMA)) < TOL


@pytest.mark.parametrize("n3f", [4, 33])
@pytest.mark.parametrize("case", ["nl_L16", "nl_L16_ref"])
def test_fp32_form(case, n3f):
    import fdga
    from fdga import _lib as ids
    box = dict(BOX, nG=6, nK1=n3f, nK2=(2, n3f), nK3=(2, n3f), mPinu=1)
    S, _ = make_pair(case, seed=11, box=box, precision="fp32")
    D, _ = make_pair(case, seed=11, box=box)
    fdga.iterate_solver(S, "fdPA")   # takes the K3 arrays into their FP32 form
    fdga.SDE(S, "fdPA")
    sigma = S.get(ids.SIGMA)
    for i in (ids.G, ids.PI0PP, ids.PI0PH, ids.PIPP, ids.PIPH):
        D.set(i, S.get(i))
    for ch in range(3):
        for cls in (1, 2, 3):
            D.set_vertex(0, ch, cls, S.vertex(0, ch, cls))
    fdga.SDE(D, "fdPA")
    assert relerr(sigma, D.get(ids.SIGMA)) < TOL
