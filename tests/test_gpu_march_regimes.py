"""Both slab regimes of the implicit-Euler march at the edges of every size bucket
and at the shortest contours, one bucket at a time, with the regime itself checked
by the bytes of the slabs that the launch keeps.

A batch keeps every fourth slab where their traffic at 5 TB/s takes over 1.6 times
its longest chain of steps; the counts here are twice what that needs if every
workgroup were resident at once.  The largest instances go through <8, 8> with 8
waves' edge values per kept slab.

Bars: extended precision, 2 N (4 + sqrt(ell)) 2^-53 as in the march's accuracy
tests.  A recomputed slab starts from a kept one, so its roundings are those of
the same N steps."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import instance, unknowns

pytestmark = pytest.mark.gpu

CAPS = [64, 128, 256, 512, 1024, 2048, 4096]


def _chain_us(cap):
    """A step of the bucket's untuned variant with the chip full."""
    K = min(8, cap // 64)
    W = cap // 64 // K
    return 0.125 + 0.02 * K + (0.1 + 0.03 * W if W > 1 else 0.0)


def _make(n, N, bc):
    it = instance(n if bc == O.BC_DN else n + 1, 2.0 + n % 5, N, bc=bc, seed=n)
    it["w"][0] = 0.0
    if bc == O.BC_DD:
        it["w"][-1] = 0.0
    q = O.march_ld(it["x"], it["w"], N, bc=bc).astype(np.longdouble)
    c = O.romberg_weights(N).astype(np.longdouble)
    it["truth"] = unknowns((c[:, None] * q * q[::-1]).sum(axis=0), bc)
    ell = max(1.0, N ** -0.5 / np.diff(it["x"]).min())
    it["tol"] = 2.0 * N * (4.0 + ell ** 0.5) * 2.0 ** -53
    return it


@pytest.mark.parametrize("every", [1, 4])
@pytest.mark.parametrize("N", [16, 32, 128])
@pytest.mark.parametrize("bc", [O.BC_DD, O.BC_DN])
@pytest.mark.parametrize("cap", CAPS)
def test_kept_slabs(cap, bc, N, every):
    import scft_amd as S
    lo = cap // 2 + 1  # (smaller ones: the shared launch below)
    sizes = [lo, lo + 1, (lo + cap) // 2 | 1, cap - 1, cap]
    mean = sum(sizes) / len(sizes)
    # slab traffic over the chain, per instance: 8 n (N - 2) bytes at 5 TB/s
    per = 8.0 * mean * (N - 2) / 5.0e6 / (_chain_us(cap) * N)
    count = -(-int(2.0 * 1.6 / per) // len(sizes)) if every == 4 else 1
    base = [_make(n, N, bc) for n in sizes]
    insts = base * count
    b = S.Batch([i["x"] for i in insts], [N] * len(insts), [unknowns(i["pt"], bc) for i in insts],
                bc=bc)
    w = np.concatenate([unknowns(i["w"], bc) for i in insts])
    out = b.eval(w)
    (items, _, nbytes), = b.time_buckets(w, 1)
    b.close()
    slabs = N - 2 if every == 1 else 2 * (N // 2 // 4)
    total = sum(len(unknowns(i["w"], bc)) for i in insts)
    assert (items, nbytes) == (len(insts), 8.0 * total * slabs + 40.0 * total)
    assert (out["status"] == 0).all()
    for k, it in enumerate(insts):
        err = float(np.abs(out["phi"][k] - it["truth"]).max())
        assert err <= it["tol"], (k, len(it["x"]), err, it["tol"])


def test_small_sizes_share_a_launch_that_recomputes():
    """Every size class of the launch for all instances of up to 512 unknowns, with
    enough of the largest beside it that every launch keeps every fourth slab."""
    import scft_amd as S
    bc, N = O.BC_DN, 64
    ns = [2, 3, 31, 63, 64, 65, 100, 127, 128, 129, 200, 255, 256, 257, 400, 511, 512, 513, 1000,
          1500]
    base = [_make(n, N, bc) for n in ns]
    big = _make(4095, N, bc)
    insts = base + [big] * 800
    b = S.Batch([i["x"] for i in insts], [N] * len(insts), [unknowns(i["pt"], bc) for i in insts],
                bc=bc)
    w = np.concatenate([unknowns(i["w"], bc) for i in insts])
    out = b.eval(w)
    rows = b.time_buckets(w, 1)
    b.close()
    n_of = np.array([len(i["x"]) - 1 for i in insts])
    edges = [0, 64, 128, 256, 512, 1024, 2048, 4096]
    want = []
    for lo, hi in zip(edges, edges[1:]):
        n = n_of[(n_of > lo) & (n_of <= hi)]
        want.append((len(n), (8.0 * 2 * (N // 2 // 4) + 40.0) * n.sum()))
    assert [(r[0], r[2]) for r in rows] == want
    assert (out["status"] == 0).all()
    for k, it in enumerate(insts):
        err = float(np.abs(out["phi"][k] - it["truth"]).max())
        assert err <= it["tol"], (k, len(it["x"]), err, it["tol"])
