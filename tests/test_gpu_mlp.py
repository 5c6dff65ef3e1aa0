"""GPU tests of the warm-start network's kernels (pecs_mlp_*): FP32 loss and
gradients against the NumPy reference (tests/mlp_reference.py, itself pinned
by finite differences), Adam training lowering the loss, BF16 inference
against FP32 inference, and the rejection of bad sizes."""
import numpy as np
import pytest

import pecs_amd
from mlp_reference import forward, layout, loss_and_grad

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


# (nin, nhidden, nlayers, nout, batch): tile edges and non-multiples of 64 / 16
@pytest.mark.parametrize("dims", [(4, 16, 3, 24, 5), (3, 70, 2, 130, 67), (4, 64, 3, 1000, 33)])
def test_gradients_match_reference(dims):
    nin, nh, nl, nout, b = dims
    _say(f"[gpu] mlp gradients {dims}")
    net = pecs_amd.WarmStartNet(nin, nh, nl, nout, seed=3)
    rng = np.random.default_rng(11)
    x = rng.normal(size=(b, nin)).astype(np.float32)
    y = rng.normal(size=(b, nout)).astype(np.float32)
    p = net.params().astype(np.float64)
    lay, npar = layout(nin, nh, nl, nout)
    assert npar == net.nparams
    loss, g = net.gradients(x, y)
    rloss, rg = loss_and_grad(p, lay, x, y)
    assert abs(loss - rloss) <= 1e-5 * abs(rloss)
    scale = np.abs(rg).max()
    assert np.abs(g - rg).max() <= 1e-4 * scale, np.abs(g - rg).max() / scale
    # FP32 inference against the reference forward pass
    yp = net.predict(x, bf16=False)
    yr = forward(p, lay, x)[-1]
    assert np.abs(yp - yr).max() <= 1e-5 * np.abs(yr).max()
    net.close()


def test_training_and_bf16_inference():
    _say("[gpu] mlp training + bf16 inference")
    rng = np.random.default_rng(2)
    nin, nout = 4, 200
    A = rng.normal(size=(nin, nout))
    x = rng.uniform(-1, 1, size=(256, nin)).astype(np.float32)
    y = (np.tanh(x @ A) + 0.1 * x[:, :1]).astype(np.float32)
    net = pecs_amd.WarmStartNet(nin, 64, 3, nout, seed=1)
    first = net.train_step(x[:64], y[:64], 3e-3)
    loss = first
    for it in range(300):
        i = (it * 64) % 256
        loss = net.train_step(x[i:i + 64], y[i:i + 64], 3e-3)
    assert loss < 0.1 * first, (first, loss)
    y32 = net.predict(x, bf16=False)
    y16 = net.predict(x, bf16=True)
    rel = np.abs(y16 - y32).max() / np.abs(y32).max()
    assert 0 < rel < 3e-2, rel   # BF16 weights and activations: a few 1e-3
    # the same after parameters are replaced (the BF16 copy is refreshed)
    p = net.params()
    net.set_params(p * 0.5)
    assert not np.allclose(net.predict(x, bf16=True), y16)
    net.close()


def test_rejects_bad_sizes():
    with pytest.raises(RuntimeError, match="sizes"):
        pecs_amd.WarmStartNet(0, 8, 2, 4)


# Large minibatches: from 512 whole 64 x 64 tiles on (256 for the input
# gradients) the dense products change kernel.  Both add their products in the
# same order, so a prediction's rows have the bits of a small batch's, with the
# same hidden units on, and the gradient is the batch-weighted mean of the
# small batches' up to the rounding of its sums: about sqrt(K) eps of their
# largest, 1.3e-5 at K = 10947 rows; bar 2e-5 of each block's largest.
@pytest.mark.parametrize("dims,rows", [((4, 256, 2, 70), (4096, 4163, 8191, 8192, 8197)), ((5, 200, 2, 64), (10943, 10947))])
def test_large_batches_match_small_ones(dims, rows):
    nin, nh, nl, nout = dims
    net = pecs_amd.WarmStartNet(nin, nh, nl, nout, seed=6)
    lay, _ = layout(nin, nh, nl, nout)
    rng = np.random.default_rng(13)
    x = rng.normal(size=(max(rows), nin)).astype(np.float32)
    y = rng.normal(size=(max(rows), nout)).astype(np.float32)
    step = 1000  # (4 x 16 tiles of 64 x 64: the small kernel)
    parts = {bf: np.concatenate([net.predict(x[i:i + step], bf16=bf) for i in range(0, len(x), step)])
             for bf in (False, True)}
    for b in rows:
        _say(f"[gpu] mlp large batch {dims} rows {b}")
        for bf in (False, True):
            assert np.array_equal(net.predict(x[:b], bf16=bf), parts[bf][:b]), (b, bf)
        loss, g = net.gradients(x[:b], y[:b])
        rloss, rg = 0.0, 0.0
        for i in range(0, b, step):
            n = min(step, b - i)
            pl, pg = net.gradients(x[i:i + n], y[i:i + n])
            rloss, rg = rloss + pl * (n / b), rg + pg.astype(np.float64) * (n / b)
        assert abs(loss - rloss) <= 1e-5 * rloss
        for lo, hi in [(w[0], w[0] + w[1] * w[2]) for w, _ in lay] + [(v[0], v[0] + v[1]) for _, v in lay]:
            d = np.abs(g[lo:hi] - rg[lo:hi]).max() / np.abs(rg[lo:hi]).max()
            assert d <= 2e-5, (b, lo, hi, d)
    net.close()


# The weight gradients of a large minibatch are summed in slices: one chain of
# n terms of one sign is off by about 0.41 u sqrt(n / 3) (u = 2^-24 half a unit
# in the last place, partial sums growing evenly), 2.6e-6 for 32768 terms added
# one by one and up to 4 times that at the worst of 4096 entries; slices of
# 1024 rows and their sum give 4.6e-7.  Bar: 6 times that, 2.8e-6, of every
# entry (targets far below the outputs, so that no term changes sign).
def test_weight_gradients_of_many_rows():
    nin, nh, nl, nout, b = 4, 64, 2, 64, 32768
    _say(f"[gpu] mlp weight gradients over {b} rows")
    net = pecs_amd.WarmStartNet(nin, nh, nl, nout, seed=8)
    rng = np.random.default_rng(14)
    x = rng.uniform(0.5, 1.5, size=(b, nin)).astype(np.float32)
    y = rng.uniform(-101, -99, size=(b, nout)).astype(np.float32)
    lay, _ = layout(nin, nh, nl, nout)
    _, rg = loss_and_grad(net.params().astype(np.float64), lay, x, y)
    _, g = net.gradients(x, y)
    (lo, fi, fo), _ = lay[-1]
    g, rg = g[lo:lo + fi * fo].reshape(fi, fo), rg[lo:lo + fi * fo].reshape(fi, fo)
    on = np.abs(rg).max(axis=1) > 1e-2 * np.abs(rg).max()  # (units that hardly ever turn on sum little)
    assert on.sum() >= nh // 4
    err = np.abs(g[on] / rg[on] - 1.0).max()
    assert err <= 2.8e-6, err
    net.close()


# encoder + convolutional decoder: (nin, nh, nl, c0, g0, stages, batch); the
# shapes cross tile edges (64-row / 64-column tiles, 16-deep k steps)
DECODERS = [
    (4, 16, 2, 4, 2, [(8, 1), (3, 0)], 3),
    (4, 40, 3, 8, 4, [(16, 1), (8, 1), (4, 0)], 5),
    (3, 24, 2, 5, 3, [(7, 1), (6, 1), (2, 1)], 2),
    (4, 32, 2, 8, 4, [(8, 1), (8, 1), (2, 1)], 16),  # weight gradients with split k (K = 16 x 32^2)
]


@pytest.mark.parametrize("spec", DECODERS)
def test_decoder_gradients_match_reference(spec):
    from mlp_reference import forward_decoder, layout_decoder, loss_and_grad_decoder
    nin, nh, nl, c0, g0, stages, b = spec
    _say(f"[gpu] decoder gradients {spec}")
    net = pecs_amd.WarmStartNet(nin, nh, nl, 0, seed=4, decoder=(c0, g0, stages))
    lay, npar = layout_decoder(nin, nh, nl, c0, g0, stages)
    assert npar == net.nparams
    G = g0 * 2 ** sum(u for _, u in stages)
    assert net.nout == stages[-1][0] * G * G
    rng = np.random.default_rng(12)
    x = rng.normal(size=(b, nin)).astype(np.float32)
    y = rng.normal(size=(b, net.nout)).astype(np.float32)
    p = net.params().astype(np.float64)
    loss, g = net.gradients(x, y)
    rloss, rg = loss_and_grad_decoder(p, lay, x, y)
    assert abs(loss - rloss) <= 1e-5 * abs(rloss)
    # per parameter block: every layer's weights and biases
    for yl in lay["layers"]:
        for lo, hi in ((yl["w"], yl["b"]), (yl["b"], yl["b"] + (yl["cout"] if yl["conv"] else yl["nout"]))):
            scale = np.abs(rg[lo:hi]).max()
            assert np.abs(g[lo:hi] - rg[lo:hi]).max() <= 1e-4 * scale + 1e-12, (yl, lo, hi)
    yp = net.predict(x, bf16=False)
    yr = forward_decoder(p, lay, x)[-1].reshape(b, -1)
    assert np.abs(yp - yr).max() <= 1e-5 * np.abs(yr).max()
    y16 = net.predict(x, bf16=True)
    rel = np.abs(y16 - yr).max() / np.abs(yr).max()
    assert 0 < rel < 3e-2, rel
    net.close()


def test_decoder_training():
    _say("[gpu] decoder training")
    rng = np.random.default_rng(7)
    G = 16
    yy, xx = np.meshgrid(np.arange(G) / G, np.arange(G) / G, indexing="ij")
    x = rng.uniform(-1, 1, size=(128, 3)).astype(np.float32)
    # smooth fields whose shape depends on the inputs
    y = np.stack([np.sin(np.pi * (xx[None] * (1 + 0.5 * x[:, :1, None]) + 0.3 * x[:, 1:2, None])) *
                  np.cos(np.pi * yy[None] * (1 + 0.3 * x[:, 2:3, None])),
                  np.exp(-((xx[None] - 0.5 - 0.2 * x[:, :1, None]) ** 2 + (yy[None] - 0.5) ** 2) * 8)], 1)
    y = y.reshape(128, -1).astype(np.float32)
    net = pecs_amd.WarmStartNet(3, 64, 2, 0, seed=2, decoder=(16, 4, [(16, 1), (2, 1)]))
    first = net.train_step(x[:32], y[:32], 2e-3)
    loss = first
    for it in range(400):
        i = (it * 32) % 128
        loss = net.train_step(x[i:i + 32], y[i:i + 32], 2e-3)
    assert loss < 0.1 * first, (first, loss)
    net.close()
