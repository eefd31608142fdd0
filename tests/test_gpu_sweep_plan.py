"""What the plan of a batch's sweep promises beyond its results: its scratch and
the slabs it keeps."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from tests.helpers import instance, unknowns

pytestmark = pytest.mark.gpu

BC = O.BC_DN


def _batch(S, parts, stepper=0, tune_file=None):
    """parts: (unknowns, steps, count); the batch, its field and one instance of each part."""
    base = [instance(n, 4.0, N, bc=BC, seed=n) for n, N, _ in parts]
    for it in base:
        it["w"][0] = 0.0
    insts = [it for it, (_, _, c) in zip(base, parts) for _ in range(c)]
    b = S.Batch([i["x"] for i in insts], [i["N"] for i in insts], [i["pt"][1:] for i in insts],
                bc=BC, stepper=stepper, tune_file=tune_file)
    return b, np.concatenate([i["w"][1:] for i in insts]), base


def _free(S):
    free, total = C.c_size_t(), C.c_size_t()
    assert S.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_scratch_of_many_small_instances_beside_a_few_larger():
    """2048 instances of 60 unknowns and 4096 steps need 2.1 GB of slabs; one
    instance of 400 in the same launch would give each of their workgroups a
    region of its size, 17 GB in all."""
    import scft_amd as S
    parts = [(60, 4096, 2048), (100, 64, 1), (200, 64, 1), (400, 4096, 1), (900, 64, 1)]
    before = _free(S)
    b, w, base = _batch(S, parts)
    used = before - _free(S)
    out = b.eval(w)
    b.close()
    assert used < 1.25 * 2.2e9 + 4.5e9, f"{used / 1e9:.1f} GB"
    assert (out["status"] == 0).all()
    k = 0
    for it, (_, N, c) in zip(base, parts):
        ref = O.evaluate(it["x"], it["w"], it["pt"], N, bc=BC)
        for j in (k, k + c - 1):
            np.testing.assert_allclose(out["phi"][j], unknowns(ref["phi"], BC), rtol=0, atol=1e-10)
        k += c


def test_tuning_does_not_change_which_slabs_are_kept():
    """One workgroup per CU (as a candidate of the autotuner, or from a tune file)
    makes the launch longer, not its slab traffic: the slabs kept follow from the
    sizes alone, and so do the bytes that time_buckets reports."""
    import tempfile

    import scft_amd as S
    parts = [(100, 64, 6000)]
    kept = 6000 * (8.0 * 100 * 2 * (64 // 2 // 4) + 40.0 * 100)
    with tempfile.NamedTemporaryFile("w", suffix=".txt") as f:
        f.write("128 2 1 1\n")
        f.flush()
        for tune in (None, f.name):
            b, w, _ = _batch(S, parts, tune_file=tune)
            (items, _, nbytes), = b.time_buckets(w, 1)
            b.close()
            assert (items, nbytes) == (6000, kept), tune
