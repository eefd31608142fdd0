"""phi of the device marches against extended precision, at bars far below the
parity tests': what the setups carry in double-double is only seen there.

The scan march (implicit Euler) takes D and A as rounded to FP64, as the
oracle's extended march does.  What is left are the roundings of the marched
rows: per step a few of its own (4 units) and those of the rows of the inverse,
one per row and independent, summed over the ell = sqrt(dt) / h rows that a row
of the inverse reaches (sqrt(ell) units).  They add up over N steps, twice in
phi = sum q q:  2 N (4 + sqrt(ell)) 2^-53.

The dense march assembles in double-double and squares with a remainder, so its
reference assembles in extended precision too, and N counts once per block of 64
steps, plus the six doublings of the first block: 4 (N / 64 + 6) units, twice."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import instance, unknowns

pytestmark = pytest.mark.gpu

LD = np.longdouble


def _make(n, N, bc, graded, cmat=O.C_ROWSCALED):
    it = instance(n if bc == O.BC_DN else n + 1, 3.72, N, bc=bc, seed=n, graded=graded)
    if cmat == O.C_ROWSCALED:
        it["w"][0] = 0.0
        if bc == O.BC_DD:
            it["w"][-1] = 0.0
    return it


def _density(q, N):
    """sum_j c_j q_j q_{N-j} of the rows q_0 .. q_N, in extended precision."""
    c = O.romberg_weights(N).astype(LD)
    q = np.asarray(q, dtype=LD)
    return (c[:, None] * q * q[::-1]).sum(axis=0)


def _device(it, N, bc, cmat=O.C_ROWSCALED, stepper=O.STEP_IE, count=1):
    import scft_amd as S
    b = S.Batch([it["x"]] * count, [N] * count, [unknowns(it["pt"], bc)] * count, bc=bc,
                cmat=cmat, stepper=stepper)
    if cmat == O.C_CONSISTENT:
        b.set_walls([it["w"][0]] * count, [it["w"][-1]] * count)
    out = b.eval([unknowns(it["w"], bc)] * count)
    b.close()
    assert (out["status"] == 0).all()
    return out["phi"][-1]


@pytest.mark.parametrize("N", [16, 64, 128, 1024])
@pytest.mark.parametrize("n", [100, 200, 400, 512, 900, 1024, 2047, 4095])
@pytest.mark.parametrize("bc,graded", [(O.BC_DD, None), (O.BC_DN, None), (O.BC_DN, 0.2)])
def test_scan_march(n, N, bc, graded):
    it = _make(n, N, bc, graded)
    truth = unknowns(_density(O.march_ld(it["x"], it["w"], N, bc=bc), N), bc)
    ell = max(1.0, N ** -0.5 / np.diff(it["x"]).min())
    tol = 2.0 * N * (4.0 + ell ** 0.5) * 2.0 ** -53
    err = float(np.abs(_device(it, N, bc) - truth).max())
    print(f"n={n} N={N} bc={bc} graded={graded}: {err:.1e} of {tol:.1e}")
    assert err <= tol


def _rows(it, N, bc, cmat):
    """Diagonals (below, on, above) of A and of dt (B + C) on the unknowns, in
    extended precision (scft.cc:641-651, 1D_FEM.c:84-186)."""
    x, w = it["x"].astype(LD), it["w"].astype(LD)
    M, dt = len(x), LD(1) / LD(N)
    u = np.arange(1, M - 1 if bc == O.BC_DD else M)
    right = u + 1 < M
    hl = x[u] - x[u - 1]
    hr = np.where(right, x[np.minimum(u + 1, M - 1)] - x[u], LD(0))
    inv = np.where(right, LD(1) / np.where(right, hr, LD(1)), LD(0))
    A = [hl / 6, hl / 3 + hr / 3, hr / 6]
    B = [-1 / hl, 1 / hl + inv, -inv]
    wi, wl, wr = w[u], w[u - 1], np.where(right, w[np.minimum(u + 1, M - 1)], LD(0))
    if cmat == O.C_ROWSCALED:
        C = [wi * a for a in A]
    else:
        C = [hl * (wl + wi) / 12, hl * (wl + 3 * wi) / 12 + hr * (3 * wi + wr) / 12,
             hr * (wi + wr) / 12]
    D = [dt * (b + c) for b, c in zip(B, C)]
    for m in (A, D):
        m[0][0] = 0
        m[2][-1] = 0
    return A, D


def _solve(lo, di, up, rhs):
    """Tridiagonal solve of the columns of rhs, by elimination."""
    n = len(di)
    di, rhs = di.copy(), rhs.copy()
    for i in range(1, n):
        f = lo[i] / di[i - 1]
        di[i] -= f * up[i - 1]
        rhs[i] -= f * rhs[i - 1]
    rhs[-1] /= di[-1]
    for i in range(n - 2, -1, -1):
        rhs[i] = (rhs[i] - up[i] * rhs[i + 1]) / di[i]
    return rhs


def _full(d):
    n = len(d[1])
    m = np.zeros((n, n), dtype=LD)
    i = np.arange(n)
    m[i, i] = d[1]
    m[i[1:], i[:-1]] = d[0][1:]
    m[i[:-1], i[1:]] = d[2][:-1]
    return m


@pytest.mark.parametrize("n,N,bc,cmat,graded,stepper", [
    (16, 256, O.BC_DD, O.C_ROWSCALED, None, O.STEP_IE),
    (31, 2048, O.BC_DD, O.C_ROWSCALED, None, O.STEP_IE),
    (32, 4096, O.BC_DN, O.C_CONSISTENT, 0.3, O.STEP_IE),
    (59, 2048, O.BC_DN, O.C_ROWSCALED, None, O.STEP_IE),
    (64, 1024, O.BC_DD, O.C_CONSISTENT, 0.3, O.STEP_IE),
    (31, 512, O.BC_DD, O.C_CONSISTENT, None, O.STEP_IRK4),
    (60, 1024, O.BC_DN, O.C_CONSISTENT, None, O.STEP_IRK4)])
def test_dense_march(n, N, bc, cmat, graded, stepper):
    it = _make(n, N, bc, graded, cmat)
    A, D = _rows(it, N, bc, cmat)
    if stepper == O.STEP_IE:
        T = _solve(A[0] + D[0], A[1] + D[1], A[2] + D[2], _full(A))
    else:  # S z = -dt D' e_k with S = A + lambda dt D', T e_k = e_k + Re((1 - i sqrt3) z)
        root3 = np.sqrt(LD(3))
        lam = LD(0.25) + 1j * (root3 / 12)
        z = _solve(*(a + lam * d for a, d in zip(A, D)), -_full(D).astype(np.clongdouble))
        T = np.eye(n, dtype=LD) + z.real + root3 * z.imag
    q = np.ones((N + 1, n), dtype=LD)
    for j in range(N):
        q[j + 1] = T @ q[j]
    tol = 2.0 * 4.0 * (N / 64 + 6) * 2.0 ** -53
    err = float(np.abs(_device(it, N, bc, cmat, stepper) - _density(q, N)).max())
    print(f"n={n} N={N}: {err:.1e} of {tol:.1e}")
    assert err <= tol
