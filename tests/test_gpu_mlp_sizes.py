"""The MLP kernels at the edges of their work split: 16-element tiles, at most
1024 work-groups with one partial-gradient row each, rows added up 128 at a
time, and the inference's element tiles.

One sample's target is far off the others', so that it alone makes most of the
gradient: whichever tile, group or row it lies in, losing it or counting it
twice moves the gradient by far more than the tolerance, 3 % of its norm (the
BF16 rounding of activations whose FP32 sums differ from the oracle's exact
ones, as in the other MLP tests)."""
import numpy as np
import pytest

import opendynamo_amd as od
from oracle import mlp as M

pytestmark = pytest.mark.gpu


def network(seed):
    rng = np.random.default_rng(seed)
    p = rng.uniform(-0.25, 0.25, od.MLP_PARAMS).astype(np.float32)
    shift = rng.uniform(-0.5, 0.5, od.MLP_FEATURES).astype(np.float32)
    scale = rng.uniform(0.5, 2.0, od.MLP_FEATURES).astype(np.float32)
    return p, shift, scale


# one sample, a ragged tile, whole tiles, a tile and one sample; 127, 128 and
# 129 partial rows; 1024 groups of one tile, and of two with a ragged last one
@pytest.mark.parametrize("n", [1, 15, 16, 17, 127 * 16, 128 * 16, 128 * 16 + 1, 1024 * 16, 1024 * 16 + 1])
def test_gradient_at_the_edges_of_the_work_split(n):
    p, shift, scale = network(n)
    rng = np.random.default_rng(n + 1)
    x = rng.standard_normal((n, od.MLP_FEATURES)).astype(np.float32)
    with od.MLP(params=p) as m:
        m.set_scaling(shift, scale)
        for at in sorted({0, n // 2, n - 1}):
            print(f"CASE test=mlp_edges n={n} at={at}", flush=True)
            t = rng.uniform(0.0, 1.0, n).astype(np.float32)
            t[at] = 4.0 * n
            loss, g = m.loss_grad(x, t)
            wl, wg = M.loss_grad(p, x, t, shift, scale)
            assert abs(loss - wl) < 0.01 * wl
            assert np.linalg.norm(g - wg) < 0.03 * np.linalg.norm(wg), (n, at)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 2048 * 16 + 1])
def test_forward_at_the_edges_of_the_work_split(n):
    p, shift, scale = network(n)
    x = np.random.default_rng(n).standard_normal((n, od.MLP_FEATURES)).astype(np.float32)
    print(f"CASE test=mlp_forward_edges n={n}", flush=True)
    with od.MLP(params=p) as m:
        m.set_scaling(shift, scale)
        y = m.forward(x)
    want, _ = M.forward(p, x, shift, scale)
    assert np.max(np.abs(y - want)) < 0.02 * np.max(np.abs(want))


# one sample, fewer samples than a batch, ragged batches, one batch per sample
@pytest.mark.parametrize("n,batch", [(1, 64), (40, 64), (1000, 300), (5, 1)])
def test_epochs_in_flight_keep_their_order_and_losses(n, batch):
    """Two epochs are in flight at a time: a run of e epochs has the losses of
    the first e epochs of a longer one, byte for byte, and its first loss is
    that of the starting weights (one batch: to f32 rounding of the sum)."""
    p, shift, scale = network(n)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, od.MLP_FEATURES)).astype(np.float32)
    t = rng.uniform(0.0, 1.0, n).astype(np.float32)
    runs = {}
    for epochs in (1, 2, 3, 6):
        print(f"CASE test=epochs n={n} batch={batch} epochs={epochs}", flush=True)
        with od.MLP(params=p) as m:
            m.set_scaling(shift, scale)
            first, _ = m.loss_grad(x, t)
            runs[epochs] = m.train(x, t, epochs=epochs, batch=batch, lr=1e-3, seed=4)
    assert len(np.unique(runs[6])) == 6
    for epochs in (1, 2, 3):
        assert runs[epochs].tobytes() == runs[6][:epochs].tobytes()
    if batch >= n:
        assert abs(runs[1][0] - first) <= 1e-5 * first
