"""The fused FP32 contraction against the FP64 one from the same state, and its persistent grids bit for bit, at every
tile count and with ragged boxes.

Tolerance: inputs rounded to 2^-24 = 6e-8, sums of at most 96 products with two operand roundings and one of the running
sum each, of random sign: some 3e-7 of the largest element a product, two products deep and with the weights 2 and -1 of
the t channel below 1e-6; a rounding in a wrong place (a sum of FP32 terms that belongs in FP64) adds one such part to
every element, a dropped term far more: 2e-6."""
import numpy as np
import pytest

from helpers import relerr
from test_gpu_bse3 import _solver

pytestmark = pytest.mark.gpu
BOXES = [(1, 2, 16), (8, 2, 16), (13, 2, 14), (24, 2, 14), (32, 2, 14), (33, 2, 14), (36, 2, 14), (40, 2, 14), (48, 2, 14)]


@pytest.mark.parametrize("nf,nb,L", BOXES)
def test_against_fp64(nf, nb, L):
    import fdga
    from fdga import _lib as ids
    A, B = (_solver(nf, nb, L, p, seed=110 + nf) for p in ("fp32", "fp64"))
    for i in (ids.PI0PP, ids.PI0PH, ids.PIPP, ids.PIPH):   # at L = 16 the FP32 solver forms the bubbles in FP32
        B.set(i, A.get(i))
    for S in (A, B):
        fdga.iterate_solver(S, "fdPA", update_Σ=False)
    for v in (0, 2):
        for ch in range(3):
            a, b = A.vertex(v, ch, 3), B.vertex(v, ch, 3)
            assert np.max(np.abs(b)) > 1e-3
            assert 0.0 < relerr(a, b) < 2e-6, (v, ch, relerr(a, b))
    A.close()
    B.close()


@pytest.mark.parametrize("nf,nb,L", [(8, 2, 16), (32, 2, 14), (36, 2, 14), (40, 2, 14), (47, 2, 14)])
def test_grids(nf, nb, L):
    import fdga
    x = []
    for grid in (0, 8, 24, 768):
        S = _solver(nf, nb, L, "fp32", seed=5)
        S.set_gemm_grid(False, grid)
        fdga.iterate_solver(S, "fdPA")
        x.append(fdga.flatten(S))
        S.close()
    for y in x[1:]:
        assert relerr(y, x[0]) == 0.0
