"""Networks that one launch takes through all layers (up to 8 layers whose
activations of 16 rows fit in LDS) and those that go layer by layer, at the
edges of the 16-wide tiles and of the 8-block ring of weight loads: outputs,
loss and gradients against the FP64 restatement, and an epoch of training
against the same batches stepped one by one."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

DIMS = [
    [1, 1],                          # one layer, one weight
    [17, 33, 16, 15],                # tile remainders
    [128, 129, 1],                   # 8 blocks of the ring, and 9
    [3, 300, 5],                     # more tiles than waves
    [20, 700, 4],                    # near the limit of LDS
    [20, 1300, 4],                   # beyond it
    [6] + [9] * 7 + [2],             # 8 layers, the most in one launch
    [6] + [9] * 8 + [2],             # 9
]


def _inputs(dims, batch):
    rng = np.random.default_rng(batch)
    return (rng.standard_normal((batch, dims[0])).astype(np.float32),
            rng.standard_normal((batch, dims[-1])).astype(np.float32))


@pytest.mark.parametrize("batch", [1, 16, 17, 67])
@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "-".join(map(str, d)))
def test_against_fp64(dims, batch):
    import scft_amd as S
    m = S.Mlp(dims, seed=11)
    p = m.params().astype(np.float64)
    p += 0.1 * np.random.default_rng(5).standard_normal(p.shape)  # biases too
    m.set_params(p.astype(np.float32))
    p = m.params().astype(np.float64)
    X, T = _inputs(dims, batch)
    # FP32 sums of K products of order 1 / sqrt(K): an error of a few 2^-24
    # sqrt(K) of the largest output; the tolerances of the 256-wide networks
    ref = O.mlp_forward(dims, p, X.astype(np.float64))
    assert np.abs(m.forward(X) - ref).max() <= 2e-5 * max(1.0, np.abs(ref).max())
    loss, g = m.loss_grad(X, T)
    lref, gref = O.mlp_loss_grad(dims, p, X.astype(np.float64), T.astype(np.float64))
    assert abs(loss - lref) <= 1e-5 * abs(lref)
    off = 0
    for l in range(len(dims) - 1):
        for n in (dims[l + 1] * dims[l], dims[l + 1]):
            a, b = g[off:off + n], gref[off:off + n]
            assert np.abs(a - b).max() <= 1e-4 * max(np.abs(b).max(), 1e-30)
            off += n
    m.close()


def _shuffled(n, seed):
    """Fisher-Yates from splitmix64(seed), as the training draws its epoch."""
    mask, idx = (1 << 64) - 1, list(range(n))
    for i in range(n - 1, 0, -1):
        seed = (seed + 0x9E3779B97F4A7C15) & mask
        z = seed
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        z ^= z >> 31
        j = z % (i + 1)
        idx[i], idx[j] = idx[j], idx[i]
    return idx


@pytest.mark.parametrize("dims", [[17, 33, 16, 15], [6] + [9] * 8 + [2]], ids=["whole", "layers"])
def test_epoch_is_its_steps(dims):
    """An epoch over 50 rows in batches of 17 (the last has 16) leaves the
    parameters that the same batches give one at a time: the same sums, so
    within rounding of each update (2^-24 of a parameter, 3 steps)."""
    import scft_amd as S
    X, T = _inputs(dims, 50)
    one, all_ = S.Mlp(dims, seed=12), S.Mlp(dims, seed=12)
    hist = all_.train(X, T, epochs=1, batch=17, lr=1e-3, seed=77)
    idx, losses = _shuffled(50, 77), 0.0
    for b in range(0, 50, 17):
        rows = idx[b:b + 17]
        loss, _ = one.loss_grad(X[rows], T[rows])
        losses += loss * len(rows)
        one.adam_step(1e-3)
    assert np.abs(all_.params() - one.params()).max() <= 1e-6
    assert abs(hist[0] - losses / 50) <= 1e-6 * hist[0]
    one.close()
    all_.close()


def test_forward_pass_of_many_rows_needs_no_training_buffers():
    """200 000 rows: the inputs, every activation and two deltas and targets as wide
    as the widest layer (a pass layer by layer) are 1.6 GB; a forward pass keeps its
    inputs and outputs."""
    import ctypes as C

    import scft_amd as S
    free, total = C.c_size_t(), C.c_size_t()
    dims, rows = [133, 256, 256, 256, 256, 136], 200000
    net = S.Mlp(dims, seed=3)
    X = np.random.default_rng(1).standard_normal((rows, dims[0])).astype(np.float32)
    assert S.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    before = free.value
    Y = net.forward(X)
    assert S.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    used = before - free.value
    assert used < 4 * rows * (sum(dims) + 2 * 256 + 136), f"{used / 1e9:.2f} GB"
    # training of fewer rows and passes of more and fewer after it keep to their buffers
    net.loss_grad(X[:50], Y[:50])
    for k in (1, 300, 7):
        np.testing.assert_array_equal(net.forward(X[-k:]), Y[-k:])
    loss, _ = net.loss_grad(X[:400], net.forward(X[:400]))
    assert loss < 1e-10  # (FP32 outputs, to their roundings)
    net.close()
