"""O.evaluate, the evaluation that device results are compared with one by one,
against the march in extended precision.

Its implicit-Euler pivots are rounded once, so what is left are the steps' own
roundings: a few units (4) per step, N steps, twice in phi, were they all of one
sign.  Pivots from the FP64 recurrence repeat a rounding over like rows, times
the rows they reach: 2e-13 to 6e-13 at these sizes, more than the margins of
1e-13 that some device tests leave for the oracle."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import instance


@pytest.mark.parametrize("m,N", [(256, 128), (1024, 64), (1024, 256), (2048, 64), (4095, 64)])
@pytest.mark.parametrize("bc", [O.BC_DD, O.BC_DN])
def test_evaluate_against_extended_precision(m, N, bc):
    it = instance(m, 3.72, N, bc=bc, seed=m)
    q = O.march_ld(it["x"], it["w"], N, bc=bc).astype(np.longdouble)
    c = O.romberg_weights(N).astype(np.longdouble)
    truth = (c[:, None] * q * q[::-1]).sum(axis=0)
    got = O.evaluate(it["x"], it["w"], it["pt"], N, bc=bc)
    assert got["rc"] == 0
    err = float(np.abs(got["phi"] - truth).max())
    tol = 2.0 * 4.0 * N * 2.0 ** -53
    print(f"m={m} N={N} bc={bc}: {err:.1e} of {tol:.1e}")
    assert err <= tol
