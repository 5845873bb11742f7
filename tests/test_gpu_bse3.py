"""BSE_L_K3! and BSE_K3! of the lattice fdPA iteration in one kernel (k_bse3) against the separate stages
(BSE_L_K3 and BSE_K3 per channel on the GEMM engine, which the oracle pins), at the K3 boxes where its tiling
can go wrong: one element, full and ragged 16 x 16 tiles, the largest box of each precision and the first
one beyond it (which takes the separate stages on both sides), on random vertices, Π's and G's.

Tolerances: FP64 sums of at most 96 terms of one magnitude differ by their order alone, some 1e-15 of the
largest element per product, two products deep: 1e-12.  FP32: the separate stages hold FL.K3 in FP64 and
round R and A alike, so the two differ by a few FP32 roundings (6e-8) of sums of at most 96 terms: 1e-5."""
import numpy as np
import pytest

from helpers import rand_c, relerr

pytestmark = pytest.mark.gpu


def _solver(nf, nb, L, precision, seed):
    import fdga
    from fdga import _lib as ids
    rng = np.random.default_rng(seed)
    nK2 = (max(nb, 2), nf)
    nK1 = max(nK2) + 1
    S = fdga.Solver(nG=nK1 + 2, nK1=nK1, nK2=nK2, nK3=(nb, nf), T=0.3, U=1.3, mPinu=2, nonlocal_=True, LG=L, L_=L,
                    ref_kind=1, ref_boxes=(nK1, nK2, (nb, nf)), precision=precision)
    Gb = fdga.hubbard_bare_Green(nK1 + 2, 0.3, L, μ=0.3, t1=1.0, t2=-0.2)
    S.set(ids.GBARE, Gb)
    S.set(ids.G0, Gb / (1.0 + Gb * rand_c(rng, Gb.shape, 0.3)))
    S.set(ids.SIGMA0, rand_c(rng, Gb.shape, 0.1))
    for v, sc in ((3, 0.3), (0, 0.2)):
        if v == 0:
            S.init()
        for ch in range(3):
            for cls in (1, 2, 3):
                S.set_vertex(v, ch, cls, rand_c(rng, S.size(ids.vertex_id(v, ch, cls)), sc))
    S.set(ids.SIGMA, rand_c(rng, Gb.size, 0.05))
    return S


def _stages(S):
    """iterate_solver!(S; strategy = :fdPA, update_Σ = false) stage by stage."""
    import fdga
    fdga.build_K3_cache(S)
    for f in (fdga.BSE_L_K2, fdga.BSE_L_K3, fdga.BSE_K1, fdga.BSE_K2, fdga.BSE_K3):
        for ch in (fdga.pCh, fdga.aCh, fdga.tCh):
            f(S, ch)
    fdga.update_F(S)


FP64 = [(1, 1, 2), (8, 2, 2), (9, 3, 2), (16, 2, 2), (17, 2, 3), (24, 2, 2), (31, 2, 2), (32, 3, 2), (33, 2, 2)]
FP32 = [(1, 2, 16), (8, 2, 16), (13, 2, 14), (23, 2, 14), (32, 2, 14), (33, 2, 14), (36, 2, 14), (40, 2, 14), (41, 2, 14),
        (48, 2, 14), (49, 2, 14)]


@pytest.mark.parametrize("precision,nf,nb,L", [("fp64",) + c for c in FP64] + [("fp32",) + c for c in FP32])
def test_one_kernel_equals_the_stages(precision, nf, nb, L):
    import fdga
    A, B = (_solver(nf, nb, L, precision, seed=100 + nf) for _ in range(2))
    tol = 1e-12 if precision == "fp64" else 1e-5
    fdga.iterate_solver(A, "fdPA", update_Σ=False)
    _stages(B)
    for v in (0, 2):
        for ch in range(3):
            a, b = A.vertex(v, ch, 3), B.vertex(v, ch, 3)
            assert np.max(np.abs(b)) > 1e-3
            assert relerr(a, b) < tol, (v, ch, relerr(a, b))
    A.close()
    B.close()


def test_persistent_grid_same_bits():
    """Workgroups looping over the (Ω, P) items give the bits of one workgroup per item."""
    import fdga
    x = []
    for grid in (0, 8, 24):
        S = _solver(9, 2, 3, "fp64", seed=5)
        S.set_gemm_grid(False, grid)
        fdga.iterate_solver(S, "fdPA")
        x.append(fdga.flatten(S))
        S.close()
    assert relerr(x[1], x[0]) == 0.0 and relerr(x[2], x[0]) == 0.0
