"""Solver groups whose members' K3 contractions run on the grouped GEMM engine, in the fused contraction, or some on each:
every tile shape and grid, the graph replay and the iterations after the autotuner give the bits of the members alone.
The autotuner leaves the solvers' state as it is, FL.K3 among it, which :scPA reads."""
import pytest

from helpers import BOX, make_pair, relerr

pytestmark = pytest.mark.gpu
TILES = ("64x64", "32x32", "64x32", "32x64")
BEYOND = dict(BOX, nK1=33, nK2=(2, 33), nK3=(2, 33), mPinu=2)   # Nν3 = 66: beyond the fused FP64 contraction


MEMBERS = {   # within the limit, beyond it, and beside each other; FP32: within it by the number of (Ω, P) pairs too
    "within": ("fp64", [("nl_L2", BOX), ("nl_L3", dict(BOX, nK3=(3, 2)))]),
    "beyond": ("fp64", [("nl_L2", BEYOND), ("nl_L3", dict(BEYOND, nK3=(1, 33)))]),
    "mixed": ("fp64", [("nl_L2", BEYOND), ("nl_L3", dict(BOX, nK3=(3, 2))), ("nl_LG4_L2", BEYOND)]),
    "mixed fp32": ("fp32", [("nl_L2", BOX), ("nl_L16_ref", dict(BOX, nK3=(2, 4)))]),
    "beyond fp32": ("fp32", [("nl_L16", dict(BOX, nK1=49, nK2=(2, 49), nK3=(2, 49), mPinu=1)), ("nl_L3", BOX)]),
}


@pytest.mark.parametrize("strategy", ["fdPA", "scPA"])
@pytest.mark.parametrize("members", list(MEMBERS))
def test_group_tiles_graph_autotune(members, strategy):
    import fdga
    precision, mem = MEMBERS[members]
    solo, grp = ([make_pair(c, seed=82 + k, box=b, precision=precision)[0] for k, (c, b) in enumerate(mem)] for _ in range(2))
    G = fdga.SolverGroup(grp)

    def step(what):
        for S in solo:
            fdga.iterate_solver(S, strategy)
        G.iterate(strategy)
        G.sync()
        for k, (a, b) in enumerate(zip(solo, grp)):
            assert relerr(fdga.flatten(b), fdga.flatten(a)) == 0.0, (what, k)

    try:
        for tile in TILES:
            for grid in (0, 8):
                G.set_tiles(0, tile, grid)
                G.set_tiles(1, tile, grid)
                step((tile, grid))
        G.set_graph(True)
        for it in range(3):
            step(("graph", it))
        G.autotune(reps=1)
        for it in range(3):
            step(("autotuned", it))
    finally:
        G.close()
