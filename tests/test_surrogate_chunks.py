"""Edges of the gradient kernel's chunks of 128 samples (tiles of 16): batches that
end inside a tile, fill a tile, fill a chunk, and give many chunks."""
import numpy as np
import pytest

import mlp_ref as M
from mytrim_amd import configs, gpu


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 20011])
def test_gradient_chunks(n):
    prob = configs.c5_c_w(10, seed=43)
    e = gpu.Engine(0)
    try:
        e.set_target(prob)
        opts = gpu.Engine.surrogate_opts(prob)
        norm = e.surrogate_norm(opts)
        rng = np.random.default_rng(n)
        p = gpu.Engine.surrogate_init(n)
        eps = np.exp(rng.uniform(np.log(norm["eps_lo"]), np.log(norm["eps_hi"]), n))
        b = norm["b_hi"] * np.sqrt(rng.random(n))
        ls2 = -8.0 + 8.0 * rng.uniform(-1.0, 1.0, n)
        g, loss = e.surrogate_grad(opts, p, eps, b, ls2)
        ref_loss, ref = M.loss_grad(p, M.inputs(norm, eps, b), M.target(norm, ls2))
        # single precision: inputs, tanh (hardware exp and reciprocal, 2 ulp) and
        # products each within 2.5e-7 relative, a chain of a dozen, 4481 sums
        assert np.linalg.norm(g - ref) <= 3e-6 * np.linalg.norm(ref) + 1e-9
        assert loss == pytest.approx(ref_loss, rel=3e-6)
        again, _ = e.surrogate_grad(opts, p, eps, b, ls2)
        assert np.array_equal(g, again)
    finally:
        e.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 17, 128, 129])
def test_gradient_with_infinite_weights(n):
    """A unit with an infinite weight is saturated: its gradient is zero, the others
    are finite, and the places of the last tile past the batch add nothing."""
    prob = configs.c5_c_w(10, seed=43)
    e = gpu.Engine(0)
    try:
        e.set_target(prob)
        opts = gpu.Engine.surrogate_opts(prob)
        norm = e.surrogate_norm(opts)
        rng = np.random.default_rng(n)
        p = gpu.Engine.surrogate_init(n)
        p[3 * 5] = np.inf    # W1: unit 5, log eps
        p[256 + 64 * 7 + 5] = -np.inf  # W2: unit 7, from unit 5
        eps = np.exp(rng.uniform(np.log(norm["eps_lo"]), np.log(norm["eps_hi"]), n))
        b = norm["b_hi"] * np.sqrt(rng.random(n))
        ls2 = -8.0 + 8.0 * rng.uniform(-1.0, 1.0, n)
        g, loss = e.surrogate_grad(opts, p, eps, b, ls2)
        # 0 times the infinite weight, in the delta of unit 5, is not a number in
        # the reference either: its own row of W1 and its bias
        with np.errstate(invalid="ignore"):
            ref_loss, ref = M.loss_grad(p, M.inputs(norm, eps, b), M.target(norm, ls2))
        assert np.array_equal(np.isfinite(g), np.isfinite(ref)) and np.isfinite(g).sum() > 4400
        ok = np.isfinite(ref)
        assert np.linalg.norm((g - ref)[ok]) <= 3e-6 * np.linalg.norm(ref[ok]) + 1e-9
        assert loss == pytest.approx(ref_loss, rel=3e-6)
    finally:
        e.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,lr", [(1000, 4e-3), (5 * 1000 + 17, 1e-30)])
def test_direct_and_replayed_epochs_agree(n, lr):
    """One epoch is launched step by step, several replay a captured one: the same
    first epoch, of one step, or of steps too small to move a weight."""
    prob = configs.c5_c_w(10, seed=43)
    out = {}
    for epochs in (1, 2, 3):
        e = gpu.Engine(0)
        try:
            e.set_target(prob)
            o = gpu.Engine.surrogate_opts(prob, n_train=n, epochs=epochs, batch=1000, lr=lr, seed=5)
            out[epochs] = e.surrogate_train(o, gpu.Engine.surrogate_init(2))
        finally:
            e.close()
    first = [r[1][0] for r in out.values()]
    assert np.isfinite(first).all() and first[0] == first[1] == first[2] > 0.0
    if lr < 1e-20:
        assert all(np.all(r[1] == first[0]) for r in out.values())
        # a bias starts at zero and moves by at most a step's size, 15 times
        assert all(np.max(np.abs(r[0] - out[1][0])) <= 1e-28 for r in out.values())
