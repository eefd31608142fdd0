"""The dense march of the smallest meshes (powers of the step matrix on the FP64
matrix cores) against the CPU oracle, for both steppers: both widths at their
smallest, odd and largest sizes, from the shortest contour that takes it, the
stored slabs as well as the density, many instances of uneven N in one launch,
and the same instances beside more buckets, where the scan march takes them.

Bars: those of the march tests, 1e-10 per stored step (relative to the step's
largest value) and on phi; the paths differ from the oracle by roundings only
(~1e-13 at these N)."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import instance, unknowns

pytestmark = pytest.mark.gpu

RTOL = ATOL = 1e-10


def _make(n, N, bc, seed, cmat=O.C_ROWSCALED, graded=None):
    it = instance(n if bc == O.BC_DN else n + 1, 2.0 + n % 5, N, bc=bc, seed=seed, graded=graded)
    if cmat == O.C_ROWSCALED:
        it["w"][0] = 0.0
        if bc == O.BC_DD:
            it["w"][-1] = 0.0
    return it


# unknowns, steps: width 32 from N = 256, width 64 from N = 512 (IRK4) or 1024
SINGLE = [(1, 256), (2, 512), (15, 256), (16, 1024), (17, 256), (31, 2048), (32, 256), (33, 1024),
          (47, 1024), (48, 2048), (63, 1024), (64, 1024), (64, 8192), (64, 512), (33, 512)]


@pytest.mark.parametrize("stepper", [O.STEP_IE, O.STEP_IRK4])
@pytest.mark.parametrize("bc,cmat", [(O.BC_DD, O.C_ROWSCALED), (O.BC_DN, O.C_CONSISTENT)])
@pytest.mark.parametrize("n,N", SINGLE)
def test_single_instance(n, N, bc, cmat, stepper):
    import scft_amd as S
    if n == 1 and bc == O.BC_DN:
        pytest.skip("a mesh of two nodes is refused")
    it = _make(n, N, bc, 40 + n, cmat, graded=0.3 if n == 48 else None)
    ref = O.evaluate(it["x"], it["w"], it["pt"], N, bc=bc, cmat=cmat, want_q=True,
                     stepper=stepper)
    assert ref["rc"] == 0
    b = S.Batch([it["x"]], [N], [unknowns(it["pt"], bc)], bc=bc, cmat=cmat, stepper=stepper)
    if cmat == O.C_CONSISTENT:
        b.set_walls([it["w"][0]], [it["w"][-1]])
    out = b.eval([unknowns(it["w"], bc)])
    assert out["status"][0] == 0
    q = b.debug_slabs(0)
    qc = ref["q"][1:N // 2]
    qc = qc[:, 1:-1] if bc == O.BC_DD else qc[:, 1:]
    assert (np.abs(q - qc).max(axis=1) / np.abs(qc).max(axis=1)).max() <= RTOL
    np.testing.assert_allclose(out["phi"][0], unknowns(ref["phi"], bc), rtol=0, atol=ATOL)
    assert abs(out["rnorm"][0] - ref["rnorm"]) <= ATOL
    again = b.eval([unknowns(it["w"], bc)])
    assert np.array_equal(out["phi"][0], again["phi"][0])
    b.close()


@pytest.mark.parametrize("stepper", [O.STEP_IE, O.STEP_IRK4])
def test_queue_and_the_scan_march_agree(stepper):
    """1500 instances (more than the grid holds) of 32 unknowns and fewer, the
    same values from one launch and, for some of them, beside four larger
    buckets (implicit Euler: the launch of the small sizes)."""
    import scft_amd as S
    kinds = [(n, N) for n in (2, 7, 16, 31, 32) for N in (1024, 2048)]
    base = [_make(n, N, O.BC_DN, 60 + n) for n, N in kinds]
    insts = [base[k % len(base)] for k in range(1500)]

    def run(insts):
        b = S.Batch([i["x"] for i in insts], [i["N"] for i in insts], [i["pt"][1:] for i in insts],
                    bc=O.BC_DN, stepper=stepper)
        out = b.eval([i["w"][1:] for i in insts])
        b.close()
        assert (out["status"] == 0).all()
        return out["phi"]

    phi = run(insts)
    for k, it in enumerate(base):
        ref = O.evaluate(it["x"], it["w"], it["pt"], it["N"], bc=O.BC_DN, stepper=stepper)
        np.testing.assert_allclose(phi[k], ref["phi"][1:], rtol=0, atol=ATOL)
    for k in range(len(insts)):
        assert np.array_equal(phi[k], phi[k % len(base)]), k
    mixed = run(base + [_make(n, 1024, O.BC_DN, 9) for n in (100, 200, 300, 900)])
    for k in range(len(base)):
        np.testing.assert_allclose(mixed[k], phi[k], rtol=0, atol=ATOL)


def test_indefinite_rows_are_flagged():
    """A field far below -1/dt: a pivot that is not positive, as in the scan march."""
    import scft_amd as S
    it = _make(20, 256, O.BC_DN, 3)
    w = it["w"][1:].copy()
    w[4:9] = -4.0 * 256
    b = S.Batch([it["x"]], [256], [it["pt"][1:]], bc=O.BC_DN)
    assert b.eval([w])["status"][0] & S.ST_PIVOT
    w[3] = np.nan
    out = b.eval([w])
    assert out["status"][0] & (S.ST_PIVOT | S.ST_NAN)
    b.close()
