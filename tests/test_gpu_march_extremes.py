"""The implicit-Euler march where the rows of D are far from 1: fields and meshes
whose units make its diagonal huge.  The rows of the inverse come from products
of the rows' determinants, which have to be rescaled before they overflow.

With a field of 1e90 everywhere D's diagonal is ~dt h 1e90 / 3, a step divides q
by more than 1e80, so phi keeps at most the c_0 q_0 q_N of that size: 0 to 1e-70
against the oracle, which eliminates row by row and never multiplies two
diagonals.  A mesh of length 1e-90 does the same through dt / h."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import instance, unknowns

pytestmark = pytest.mark.gpu

BC = O.BC_DN


@pytest.mark.parametrize("n", [2, 64, 100, 200, 400, 1000, 2000, 4096])
@pytest.mark.parametrize("what", ["field", "mesh"])
def test_huge_diagonal(n, what):
    import scft_amd as S
    N = 32  # (the dense march takes no contour this short)
    it = instance(n, 4.0, N, bc=BC, seed=n)
    x, w = it["x"], it["w"]
    if what == "field":
        w = w + 1e90
        w[0] = 0.0
    else:
        x = x * 1e-90
    ref = O.evaluate(x, w, it["pt"], N, bc=BC)
    assert ref["rc"] == 0 and np.isfinite(ref["phi"]).all()
    for count in (1, 3):
        b = S.Batch([x] * count, [N] * count, [unknowns(it["pt"], BC)] * count, bc=BC)
        out = b.eval([unknowns(w, BC)] * count)
        b.close()
        assert (out["status"] == 0).all(), out["status"]
        for phi in out["phi"]:
            np.testing.assert_allclose(phi, unknowns(ref["phi"], BC), rtol=0, atol=1e-10)


@pytest.mark.parametrize("stepper", [O.STEP_IE, O.STEP_IRK4])
@pytest.mark.parametrize("n", [20, 60, 300])
def test_huge_field_of_either_stepper(n, stepper):
    """The same through the dense march (up to 64 unknowns) and IRK4, whose step
    factor tends to 1 there: phi is that of q_j = 1."""
    import scft_amd as S
    N = 1024
    it = instance(n, 4.0, N, bc=BC, seed=n)
    w = it["w"] + 1e90
    w[0] = 0.0
    ref = O.evaluate(it["x"], w, it["pt"], N, bc=BC, stepper=stepper)
    assert ref["rc"] == 0 and np.isfinite(ref["phi"]).all()
    b = S.Batch([it["x"]], [N], [unknowns(it["pt"], BC)], bc=BC, stepper=stepper)
    out = b.eval([unknowns(w, BC)])
    b.close()
    assert out["status"][0] == 0
    np.testing.assert_allclose(out["phi"][0], unknowns(ref["phi"], BC), rtol=0, atol=1e-10)
