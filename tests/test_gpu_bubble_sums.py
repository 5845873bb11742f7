"""The lattice bubble's sums over ω: the same bits whether all of Π is stored or the band alone, and no more memory
than the chunks that they cover."""
import ctypes
import gc

import pytest

from helpers import BOX, EXTRA_CASES, make_pair, relerr

pytestmark = pytest.mark.gpu
for _L in (4, 9, 16, 24):
    EXTRA_CASES[f"sums_L{_L}"] = (True, _L, _L, 0, False)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nG", [5, 40])
@pytest.mark.parametrize("L", [4, 9, 16, 24])
def test_reading_pi_leaves_the_iteration(L, nG, precision):
    """Reading Π makes the solver recompute it in full; the next iteration on the same Σ gives the bits that it
    gives without the read (both take the same products in the same order)."""
    import fdga
    from fdga import _lib as ids
    x = []
    for read in (False, True):
        S, _ = make_pair(f"sums_L{L}", seed=4, box=dict(BOX, nG=nG, nK1=4, nK2=(2, 3), nK3=(2, 2), mPinu=16), precision=precision)
        fdga.iterate_solver(S, "fdPA")
        if read:
            S.get(ids.PIPP)
            S.get(ids.PIPH)
        fdga.iterate_solver(S, "fdPA", update_Σ=False)
        x.append(fdga.flatten(S))
        S.close()
    assert relerr(x[1], x[0]) == 0.0


def test_memory():
    """A 32 x 32 lattice whose bubble mesh is 16 times the K1 box and G's mesh: the four Π arrays are 1.04 GB, and
    all else (the sums on the chunks that meet the band or G's mesh 7 % of that) stays below a quarter of it."""
    import fdga

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert fdga.load().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    gc.collect()
    before = free()
    S = fdga.Solver(nG=16, nK1=16, nK2=(4, 4), nK3=(2, 2), T=0.3, U=1.0, mPinu=16, nonlocal_=True, LG=32, L_=32)
    used = before - free()
    pi = 4 * 16 * (2 * 16 * 16) * 31 * 32 * 32
    S.close()
    assert used < 1.25 * pi, (used, pi)
