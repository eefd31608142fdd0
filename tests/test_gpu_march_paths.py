"""The march's paths that a batch's size selects, against the CPU oracle at the
edges of their ranges:

  * every fourth slab kept and the others recomputed (batches whose slab
    traffic outlasts their longest chain of steps), one bucket at a time at its
    smallest, odd and largest sizes, and N down to the shortest contour;
  * the launch that takes all instances of up to 512 unknowns together
    (batches over more than four buckets), with and without that;
  * pairing weights by class at the smallest N.

Bar: |phi_dev - phi_cpu| <= 1e-10, the bar of the other march tests (phi is
O(1); the worst oracle error of the shapes here against extended precision is
below 2e-11)."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import instance, unknowns

pytestmark = pytest.mark.gpu

PHI_ATOL = 1e-10

# bucket capacity -> instances that put its slab traffic past its chain of steps
MANY = {64: 4500, 128: 2800, 256: 1700, 512: 1000, 1024: 700, 2048: 420, 4096: 280}


def _check(S, insts, bc):
    Ns = [it["N"] for it in insts]
    ref = O.batch_eval([it["M"] for it in insts], Ns, [it["x"] for it in insts],
                       [it["pt"] for it in insts], [it["w"] for it in insts], bc=bc)
    assert ref["rc"] == 0
    b = S.Batch([it["x"] for it in insts], Ns, [unknowns(it["pt"], bc) for it in insts], bc=bc)
    out = b.eval([unknowns(it["w"], bc) for it in insts])
    b.close()
    assert (out["status"] == 0).all()
    for k, it in enumerate(insts):
        np.testing.assert_allclose(out["phi"][k], unknowns(ref["phi"][k], bc), rtol=0,
                                   atol=PHI_ATOL, err_msg=f"instance {k} M={it['M']} N={it['N']}")
    np.testing.assert_allclose(out["rnorm"], ref["rnorm"], rtol=0, atol=PHI_ATOL)


def _make(n, N, L, bc, seed):
    it = instance(n if bc == O.BC_DN else n + 1, L, N, bc=bc, seed=seed)
    it["w"][0] = 0.0
    if bc == O.BC_DD:
        it["w"][-1] = 0.0
    return it


@pytest.mark.parametrize("bc", [O.BC_DD, O.BC_DN])
@pytest.mark.parametrize("cap", sorted(MANY))
def test_recomputed_slabs(cap, bc):
    import scft_amd as S
    lo = cap // 2 + 1 if cap > 64 else 2
    sizes = [lo, lo + 1, (lo + cap) // 2 | 1, cap - 1, cap]
    insts, base = [], {}
    for k in range(MANY[cap]):
        n, N = sizes[k % len(sizes)], (16, 32, 64)[k % 3]
        if (n, N) not in base:
            base[n, N] = _make(n, N, 2.0 + k % 5, bc, 900 + k)
        insts.append(base[n, N])
    _check(S, insts, bc)


def test_small_sizes_in_one_launch():
    """Five and more buckets: every size of up to 512 unknowns through one
    launch, every slab kept; then with 280 of the largest instances beside
    them, every fourth."""
    import scft_amd as S
    ns = [2, 3, 31, 63, 64, 65, 100, 127, 128, 129, 200, 255, 256, 257, 400, 511, 512, 513, 1000,
          1500, 4095]
    few = [_make(n, (16, 32, 256)[i % 3], 2.0 + i % 6, O.BC_DN, 300 + i) for i, n in enumerate(ns)]
    _check(S, few, O.BC_DN)
    big = _make(4095, 32, 6.0, O.BC_DN, 77)
    _check(S, few + [big] * 700, O.BC_DN)


@pytest.mark.parametrize("ns", [[100, 500], [40, 100, 200, 500, 1000]], ids=["buckets", "grouped"])
def test_some_launches_recompute(ns):
    """Slab traffic between the two regimes: the launches of small instances
    keep every fourth slab, the one large instance, the longest chain, all."""
    import scft_amd as S
    bc = O.BC_DN
    base = [_make(n, 64, 3.0, bc, n) for n in ns]
    big = _make(4095, 128, 6.0, bc, 7)
    mean = sum(ns) / len(ns)
    count = int(0.7 * 80.0 * 5.0e6 / (8.0 * mean * 64)) // len(ns)  # 0.7 of ~80 us at 5 TB/s
    insts = base * count + [big]
    _check(S, insts, bc)
    b = S.Batch([it["x"] for it in insts], [it["N"] for it in insts],
                [unknowns(it["pt"], bc) for it in insts], bc=bc)
    times = b.time_buckets(b.join([unknowns(it["w"], bc) for it in insts]), 1)
    b.close()
    for (items, _, nbytes), it in zip(times, base + [big]):
        n, N = len(it["x"]) - 1, it["N"]
        kept = 8.0 * n * (N - 2) if it is big else 8.0 * n * 2 * (N // 8)
        assert nbytes == items * (kept + 40.0 * n)


@pytest.mark.parametrize("N", [16, 32, 64, 128])
def test_pairing_weights_by_class(N):
    import scft_amd as S
    _check(S, [_make(40, N, 3.0, O.BC_DD, 5)], O.BC_DD)


@pytest.mark.parametrize("n", [257, 511, 512, 513, 1000, 1024])
def test_irk4_rows_per_lane(n):
    """IRK4 buckets of 512 and 1024 unknowns take four rows per lane while every
    instance finds a CU, eight beyond."""
    import scft_amd as S
    bc, cmat, N = O.BC_DN, O.C_CONSISTENT, 32
    it = _make(n, N, 4.0, bc, n)
    ref = O.evaluate(it["x"], it["w"], it["pt"], N, bc=bc, cmat=cmat, stepper=O.STEP_IRK4)
    for count in (1, 700):
        b = S.Batch([it["x"]] * count, [N] * count, [unknowns(it["pt"], bc)] * count, bc=bc, cmat=cmat,
                    stepper=S.STEP_IRK4)
        out = b.eval([unknowns(it["w"], bc)] * count)
        b.close()
        assert (out["status"] == 0).all()
        for phi in out["phi"]:
            np.testing.assert_allclose(phi, unknowns(ref["phi"], bc), rtol=0, atol=PHI_ATOL)
