"""The lattice bubble where its inner range and its direct transform can go wrong: the smallest lattices, L with
four outputs a thread left over, the largest L of a single ω per block; G's mesh narrower than the band, between
band and mesh, and wider than the mesh (no sums beyond the inner range); a finer momentum mesh of G.  The whole of
Π (read back after an iteration that stored the band only), and an iteration that takes the far sums, against the
oracle: sums of at most 4 L² products of order one, for which 1e-12 is over ten times the rounding."""
import pytest

import pyoracle as po
from helpers import BOX, EXTRA_CASES, make_pair, relerr

pytestmark = pytest.mark.gpu
TOL = 1e-12
for _L, _f in ((1, 1), (2, 1), (7, 1), (9, 2), (12, 1), (16, 1), (17, 1), (32, 1)):
    EXTRA_CASES[f"bubble_L{_L}"] = (True, _f * _L, _L, 0, False)
LS = [1, 2, 7, 9, 12, 16, 17, 32]


@pytest.mark.parametrize("nG", [3, 14, 40])
@pytest.mark.parametrize("L", LS)
def test_ranges(L, nG):
    import fdga
    from fdga import _lib as ids
    box = dict(BOX, nG=nG, nK1=3, nK2=(1, 2), nK3=(1, 1), mPinu=7)
    S, O = make_pair(f"bubble_L{L}", seed=5, box=box)
    fdga.iterate_solver(S, "scPA")
    O.iterate(po.SCPA)
    assert relerr(fdga.flatten(S), O.flatten()) < TOL
    for hw, ow in ((ids.PIPP, po.PIPP), (ids.PIPH, po.PIPH)):
        assert relerr(S.get(hw), O.get(ow)) < TOL
