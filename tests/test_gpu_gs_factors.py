"""The factors of the rational ground-state form, split over 256 threads: sizes
with empty chunks, one and two rows per thread, and last chunks that end inside a
wave, through one and two mixer updates against the oracle, which eliminates row
by row.

The reference is the oracle's mixer over the device's own evaluations: an update
takes second differences of log phi, so at 4096 unknowns (1 / h^2 = 1e6) a rounding
of phi alone moves it by 1e-8.

Bar: 1e-8 of each value of the field (of 1 for smaller ones), the bar of the other
mixer trajectories.  The rational part of these updates is 0.5 to 1 away from the
wall, and 1e-12 on the first field moves the oracle's result by at most 1e-9."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from scft_amd import workloads as WL

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 255, 256, 257, 511, 512, 513, 767, 1025, 4095, 4096]


def _oracle_mixer(evaluate, x, pt, N, w, bc, **kw):
    """orc_anderson of one instance; evaluate: unknowns -> residual."""
    last = -1 if bc == O.BC_DD else None
    n = len(x[1:last])

    @O.RESIDUAL_FN
    def residual(n, pw, pr, ctx):
        r = evaluate(np.ctypeslib.as_array(pw, (n,)).copy())
        np.ctypeslib.as_array(pr, (n,))[:] = r
        return 0

    ps, gs, got = np.zeros(3 * n), np.zeros(3 * n), w[1:last].copy()
    lib = O.lib()
    lib.orc_precond_stencil(x, len(x), bc, ps)
    lib.orc_gs_stencil(x, len(x), bc, gs)
    o = O.anderson_opts(**kw)
    o.field_lower = -o.field_floor * N
    o.pstencil, o.gstencil = ps.ctypes.data, gs.ctypes.data
    st = O.AndersonStats(0, 0, 0.0, None, 0)
    lib.orc_anderson(got, n, C.cast(residual, C.c_void_p), None, C.byref(o),
                     pt[1:].ctypes.data, C.byref(st))
    return got


@pytest.mark.parametrize("updates", [1, 2])
@pytest.mark.parametrize("bc", [O.BC_DD, O.BC_DN])
def test_rational_form_at_the_edges_of_its_chunks(bc, updates):
    import scft_amd as S
    dd = bc == O.BC_DD
    xs, pts, ws = [], [], []
    for n in SIZES:
        if not dd and n < 2:
            continue  # (no mesh of two nodes)
        M = n + (2 if dd else 1)
        # spacing up to twice the first cell's, shorter meshes for fewer nodes
        x = np.linspace(0.0, 1.0, M)
        x = min(3.72, 0.02 * M) * (x + x * x) / 2.0
        w = WL.w0_field(x, n)
        w[0] = 0.0
        if dd:
            w[-1] = 0.0
        xs.append(x)
        pts.append(O.target_position(x, O.TAU, dd))
        ws.append(w)
    N = 64
    last = -1 if dd else None
    kw = dict(history=8, tol=1e-30, transform=2, beta=1.0, step_cap=0.0, precond=0.5,
              field_floor=0.5, gs_precond=0.5, gs_field_weight=0.25, gs_shift=3.0)
    b = S.Batch(xs, [N] * len(xs), [p[1:last] for p in pts], bc=bc)
    out = b.solve([w[1:last] for w in ws], S.anderson_opts(max_iter=updates + 1, check_every=1, **kw))
    for k, x in enumerate(xs):
        def evaluate(w, k=k):
            fields = [v[1:last] for v in ws]
            fields[k] = w
            return b.eval(fields)["r"][k]
        want = _oracle_mixer(evaluate, x, pts[k], N, ws[k], bc, max_iter=updates, **kw)
        dw = (np.abs(out["w"][k] - want) / np.maximum(1.0, np.abs(want))).max()
        print(f"n={len(x) - (2 if dd else 1)}: |w_dev - w_cpu| = {dw:.1e}")
        assert dw <= 1e-8, len(x)
    b.close()
