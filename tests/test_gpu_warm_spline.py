"""The spline of the device-side warm start (cyclic reduction, a thread per
row of its system) against the host's elimination, from the smallest table to
the largest and around the powers of two where a step is added, on uneven
grids."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_grid", [4, 5, 6, 7, 10, 11, 66, 67, 128, 255, 256])
def test_spline_matches_host(n_grid):
    import scft_amd as S
    rng = np.random.default_rng(n_grid)
    xs = [np.concatenate([[0.0], np.sort(rng.uniform(0.0, 4.0, n - 2)), [4.0]]) for n in (9, 40, 700)]
    b = S.Batch(xs, [64] * 3, [np.ones(len(x) - 1) for x in xs], bc=S.BC_DN)
    steps = rng.uniform(1.0, 3.0, (3, n_grid - 1))
    grid = np.concatenate([np.zeros((3, 1)), np.cumsum(steps, axis=1)], axis=1)
    grid *= 4.0 / grid[:, -1:]
    net = S.Mlp([3, n_grid], seed=n_grid)
    F = rng.standard_normal((3, 3)).astype(np.float32)
    plan = S.WarmPlan(b, net, F, grid, [], 1.0, [0, 0, 0])
    plan.predict()
    w = b.download()["w"]
    y = net.forward(F).astype(np.float64)
    ref = S.resample_spline_batch(list(grid), list(y), [x[1:] for x in xs])
    for got, want in zip(w, ref):
        # rows dominated by their diagonal 3 : 2 at least, so both eliminations
        # are within a few 2^-53 of the exact solution per step of theirs
        assert np.abs(got - want).max() <= 1e-12 * max(1.0, np.abs(y).max())
    plan.close()
    b.close()
    net.close()
