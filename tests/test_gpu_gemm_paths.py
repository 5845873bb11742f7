"""The K3 contractions that stay on the batched GEMM engine or on BSE_L_K3!'s momentum-batched kernels: the stage calls,
:scPA, K3 boxes beyond the fused contraction's limit, and the FP32 mfRG map (solver groups: test_gpu_group_paths.py).
Tile shapes and persistent grids leave every bit as it is (each element accumulates over k in the same order).

FP32 against FP64 (the mfRG map): 64 products, each with two operands rounded to 2^-24 = 6e-8 and one rounding of the
running sum, of random sign, leave some 3e-7 of the largest element, two products deep; 2e-6 is over five times that."""
import numpy as np
import pytest

from helpers import BOX, make_pair, rand_c, relerr
from test_gpu_bse3 import _solver

pytestmark = pytest.mark.gpu
TILES = ("64x64", "32x32", "64x32", "32x64")
BEYOND = dict(BOX, nK1=33, nK2=(2, 33), nK3=(2, 33), mPinu=2)   # Nν3 = 66: beyond the fused FP64 contraction


def _stages(S):
    import fdga
    fdga.build_K3_cache(S)
    for f in (fdga.BSE_L_K3, fdga.BSE_K3):
        for ch in (fdga.pCh, fdga.aCh, fdga.tCh):
            f(S, ch)
    return np.concatenate([S.vertex(v, ch, 3) for v in (1, 2) for ch in range(3)])


def _settings():
    for tl in TILES:
        for tk in TILES:
            yield tl, tk, 0
    for grid in (8, 24, 192):
        yield "64x64", "64x64", grid
        yield "32x32", "64x32", grid


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case,box", [("nl_L2", BOX), ("nl_L2", BEYOND), ("nl_L16_ref", dict(BOX, nK3=(2, 4)))])
def test_stage_calls(case, box, precision):
    ref = _stages(make_pair(case, seed=80, box=box, precision=precision)[0])
    S, _ = make_pair(case, seed=80, box=box, precision=precision)
    assert np.max(np.abs(ref)) > 1e-3
    for tl, tk, grid in _settings():
        S.set_gemm_tile(True, tl)
        S.set_gemm_tile(False, tk)
        S.set_gemm_grid(True, grid)
        S.set_gemm_grid(False, grid)
        assert relerr(_stages(S), ref) == 0.0, (tl, tk, grid)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case,box,strategy", [("nl_L2", BOX, "scPA"), ("nl_L16_ref", dict(BOX, nK3=(2, 4)), "scPA"),
                                               ("nl_L2", BEYOND, "fdPA"), ("nl_L2", BEYOND, "scPA_new")])
def test_iterations(case, box, strategy, precision):
    import fdga
    ref, _ = make_pair(case, seed=81, box=box, precision=precision)
    x0 = fdga.flatten(ref)
    fdga.iterate_solver(ref, strategy)
    want = fdga.flatten(ref)
    S, _ = make_pair(case, seed=81, box=box, precision=precision)
    for tl, tk, grid in _settings():
        fdga.unflatten(S, x0)
        S.set_gemm_tile(True, tl)
        S.set_gemm_tile(False, tk)
        S.set_gemm_grid(True, grid)
        S.set_gemm_grid(False, grid)
        fdga.iterate_solver(S, strategy)
        assert relerr(fdga.flatten(S), want) == 0.0, (tl, tk, grid)


@pytest.mark.parametrize("strategy", ["fdPA", "fdPA_new"])
@pytest.mark.parametrize("nf,nb,L", [(32, 2, 14), (31, 2, 14), (9, 2, 14), (33, 2, 14)])
def test_fp32_mfrg_map(nf, nb, L, strategy):
    """The mfRG map of an FP32 lattice solver, whose BSE_L_K3! takes the momentum-batched kernels up to Nν3 = 64 (the
    software-pipelined one at 64) and the GEMMs beyond, against the FP64 solver's, before and after an iteration that
    holds K3 in FP32; and with its workgroups looping over their tasks."""
    import fdga
    S, D = (_solver(nf, nb, L, p, seed=90 + nf) for p in ("fp32", "fp64"))
    rng = np.random.default_rng(91)
    n = S.lib.fdga_flat_size_F(S.h)
    x = rand_c(rng, n, 0.3)
    y = []
    for T in (S, D):
        fdga.build_K3_cache(T)
        y.append(fdga.mfRGLinearMap(T, strategy) @ x)
    k3 = np.max(np.abs(D.vertex(2, 0, 3)))
    assert k3 > 1e-6
    assert np.max(np.abs(y[0] - y[1])) < 2e-6 * np.max(np.abs(y[1] - x)), np.max(np.abs(y[0] - y[1])) / np.max(np.abs(y[1] - x))
    for grid in (8, 64):
        S.set_gemm_grid(True, grid)
        fdga.build_K3_cache(S)
        assert relerr(fdga.mfRGLinearMap(S, strategy) @ x, y[0]) == 0.0, grid
    fdga.iterate_solver(S, "fdPA", update_Σ=False)
    fdga.build_K3_cache(S)
    z = fdga.mfRGLinearMap(S, strategy) @ x
    assert np.max(np.abs(z - y[1])) < 2e-6 * np.max(np.abs(y[1] - x))
    S.close()
    D.close()
