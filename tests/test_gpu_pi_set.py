"""One bubble array set and the other read back after an iteration that stored it on the band only: the read recomputes
the one and leaves the other as it was set, with its sums."""
import numpy as np
import pytest

from helpers import BOX, make_pair, rand_c, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", ["pp", "ph"])
@pytest.mark.parametrize("case", ["nl_L3", "local_ref"])
def test_set_then_read(case, first):
    import fdga
    from fdga import _lib as ids
    box = dict(BOX, nG=5, nK1=4, nK2=(2, 3), nK3=(2, 2), mPinu=8)
    one, other = (ids.PIPP, ids.PIPH) if first == "pp" else (ids.PIPH, ids.PIPP)
    x = []
    for read in (False, True):
        S, _ = make_pair(case, seed=6, box=box)
        fdga.iterate_solver(S, "fdPA")
        a = rand_c(np.random.default_rng(7), S.size(one), 0.2)
        S.set(one, a)
        if read:
            b = S.get(other)
            assert np.max(np.abs(b)) > 1e-3
            assert np.array_equal(S.get(one), a)
        fdga.iterate_solver(S, "fdPA", update_Σ=False)
        x.append(fdga.flatten(S))
        S.close()
    assert relerr(x[1], x[0]) == 0.0
