"""Iterations with event timing on, alone and in a group, give the bits of the untimed ones: the timed forms launch the
same kernels in another order and on other streams.  Groups with every lattice member in the fused contraction, with
some (a K3 box beyond its limit beside one within it), with none, and of local solvers."""
import pytest

from helpers import BOX, make_pair, relerr

pytestmark = pytest.mark.gpu
WIDE = dict(BOX, nK1=63, nK2=(4, 5), nK3=(3, 5), mPinu=3)        # local: K2 from copies along its diagonals
BEYOND = dict(BOX, nK1=33, nK2=(2, 33), nK3=(2, 33), mPinu=2)    # Nν3 = 66


@pytest.mark.parametrize("groups", [False, True])
@pytest.mark.parametrize("strategy", ["fdPA", "scPA", "fdPA_new"])
@pytest.mark.parametrize("case,box", [("local_ref", BOX), ("local_vertexref", WIDE), ("nl_L2", BOX), ("nl_L3", BEYOND)])
def test_solver(case, box, strategy, groups):
    import fdga
    x = []
    for timed in (False, True):
        S, _ = make_pair(case, seed=60, box=box)
        if groups:
            S.init_sym_grp()
        S.set_stage_timing(timed)
        for _ in range(2):
            fdga.iterate_solver(S, strategy)
        x.append(fdga.flatten(S))
        if timed:
            assert S.stage_ms()[6] > 0
        S.close()
    assert relerr(x[1], x[0]) == 0.0


GROUPS = {
    "all fused": ("fp64", [("nl_L2", BOX), ("nl_L3", dict(BOX, nK3=(3, 2)))]),
    "some fused": ("fp64", [("nl_L2", BOX), ("nl_L2", BEYOND), ("nl_L3", dict(BOX, nK3=(3, 2)))]),
    "none fused": ("fp64", [("nl_L2", BEYOND), ("nl_L3", BEYOND)]),
    "some fused, fp32": ("fp32", [("nl_L2", BOX), ("nl_L16", dict(BOX, nK3=(2, 4)))]),
    "local": ("fp64", [("local_ref", BOX), ("local_vertexref", WIDE)]),
}


@pytest.mark.parametrize("strategy", ["fdPA", "scPA"])
@pytest.mark.parametrize("members", list(GROUPS))
def test_group(members, strategy):
    import fdga
    precision, mem = GROUPS[members]
    x = []
    for timed in (False, True):
        S = [make_pair(c, seed=70 + k, box=b, precision=precision)[0] for k, (c, b) in enumerate(mem)]
        G = fdga.SolverGroup(S)
        try:
            G.set_timing(timed)
            for _ in range(2):
                G.iterate(strategy)
            G.sync()
            if timed:
                assert sum(G.gemm_ms()) > 0
            x.append([fdga.flatten(s) for s in S])
        finally:
            G.close()
        for s in S:
            s.close()
    for a, b in zip(*x):
        assert relerr(b, a) == 0.0
