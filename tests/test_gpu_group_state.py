"""Members of a solver group at different F/Fbuff states (one updated on its own) are refused, whichever form their
contractions take, and nothing has run then: the iteration after the states agree again is that of the members alone."""
import pytest

from helpers import BOX, make_pair, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strategy", ["fdPA", "scPA"])
@pytest.mark.parametrize("case,box", [("nl_L2", BOX), ("nl_L2", dict(BOX, nK1=33, nK2=(2, 33), nK3=(1, 33))), ("local_ref", BOX)])
def test_refused(case, box, strategy):
    import fdga
    grp = [make_pair(case, seed=50 + k, box=box)[0] for k in range(2)]
    solo = [make_pair(case, seed=50 + k, box=box)[0] for k in range(2)]
    G = fdga.SolverGroup(grp)
    try:
        fdga.update_F(grp[1])
        with pytest.raises(fdga.FdgaError, match="same iteration"):
            G.iterate(strategy)
        fdga.update_F(grp[1])
        G.iterate(strategy)
        G.sync()
        for a, b in zip(solo, grp):
            fdga.iterate_solver(a, strategy)
            assert relerr(fdga.flatten(b), fdga.flatten(a)) == 0.0
    finally:
        G.close()
