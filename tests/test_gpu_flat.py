"""The solver vector's layout change (k_unflatten, k_flatten): exact copies, so every comparison is for equal
bits.  Local, lattice with unequal boxes, and the FP32 lattice iteration, whose K3 arrays are held in FP32
(values that FP32 holds exactly survive the round trip)."""
import numpy as np
import pytest

from helpers import BOX, make_pair

pytestmark = pytest.mark.gpu
CASES = [("local_ref", BOX, "fp64"), ("nl_L3", dict(BOX, nK3=(3, 2)), "fp64"), ("nl_L2", dict(BOX, nK3=(1, 1)), "fp64"),
         ("nl_L16", dict(BOX, nK3=(2, 4)), "fp32")]


@pytest.mark.parametrize("case,box,precision", CASES)
def test_layout_and_residual(case, box, precision):
    import fdga
    from fdga import _lib as ids
    S, O = make_pair(case, seed=3, box=box, precision=precision)
    if precision == "fp32":
        fdga.iterate_solver(S, "fdPA")   # takes the K3 arrays into their FP32 form
    rng = np.random.default_rng(9)
    n = S.lib.fdga_flat_size(S.h)
    x = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64).astype(np.complex128)
    fdga.unflatten(S, x)
    assert np.array_equal(fdga.flatten(S), x)
    parts = [S.vertex(0, ch, cls) for ch in range(3) for cls in (1, 2, 3)] + [S.get(ids.SIGMA)]
    assert np.array_equal(np.concatenate(parts), x)
    x *= 0.01
    R = np.zeros_like(x)
    fdga.fixed_point(R, x, S, "fdPA")
    assert np.array_equal(R, fdga.flatten(S) - x)
    nF = S.lib.fdga_flat_size_F(S.h)
    RF = np.zeros(nF, complex)
    fdga.fixed_point(RF, x[:nF], S, "fdPA", update_Σ=False)
    assert np.array_equal(RF, fdga.flatten_vertex(S) - x[:nF])
