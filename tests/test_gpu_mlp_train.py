"""The fused training step (one kernel for the forward, the loss and the backward's chain, one for every
layer's gradients) where its tiles can go wrong: batches around the 16- and 32-sample tiles and around
the switch between one and two row tiles per workgroup, every width it is built for and the layered
path past them, one hidden layer and many, inputs and outputs that fill their padding; against the FP64
oracle of the BF16 network, whose gradients the kernels' own roundings of the activations and of dZ
leave within the bound below. And epochs of one batch and of batches that are alike against the same
batches given one by one to gradients() and adam_step(), and which samples an epoch's batches take."""

from __future__ import annotations

import numpy as np
import pytest

from autan_amd.mlp import MLP
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def data(n, d_in, d_out, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, size=(n, d_in)).astype(np.float32)
    t = np.stack([np.sin((j + 1) * x[:, j % d_in]) + x[:, (j + 2) % d_in] for j in range(d_out)], axis=1)
    return x, t.astype(np.float32)


@pytest.mark.parametrize("hidden,layers,d_in,d_out", [(64, 1, 7, 5), (128, 3, 1, 1), (192, 2, 32, 16), (256, 6, 7, 5),
                                                      (320, 2, 7, 5)])
@pytest.mark.parametrize("n", [1, 16, 17, 33, 8192, 8193])
def test_gradients_at_the_tiles_edges(hidden, layers, d_in, d_out, n):
    m = MLP(d_in, hidden, layers, d_out, seed=n)
    x, t = data(n, d_in, d_out, n + 1)
    m.fit_normalization(*data(2000, d_in, d_out, 5))
    loss, g = m.gradients(x, t)
    norm = [np.asarray(a, np.float64) for a in m.norm]
    l_o, g_o = mo.loss_and_gradients(m.params(), m.widths(), x, t, norm, d_out, bf=True)
    assert abs(loss - l_o) <= 1e-2 * l_o
    # Each BF16 rounding of a layer (2^-9 of a value) enters the gradients below it once, forward and
    # backward: 2 layers of them, uncorrelated, well under 3 % of the norm.
    at = 0
    w = m.widths()
    for l in range(len(w) - 1):
        k, nn = w[l], w[l + 1]
        for size in (nn * k, nn):
            seg = slice(at, at + size)
            at += size
            assert np.linalg.norm(g[seg] - g_o[seg]) <= 5e-2 * np.linalg.norm(g_o[seg]) + 1e-12, (l, size)
    m.close()


@pytest.mark.parametrize("hidden", [64, 256])
def test_an_epoch_is_its_batches(hidden):
    """One batch per epoch: the shuffle only permutes its samples, so the epochs' weights are those of
    gradients() and adam_step() on the batch, but for the order of FP32 sums: the gradients' relative
    difference of a few 2^-24 times the square root of the samples changes each Adam step (lr at most per
    weight, whatever the gradient's size) only where the gradient itself is that small."""
    n, steps, lr = 500, 4, 1e-3
    x, t = data(n, 7, 5, 3)
    a, b = MLP(7, hidden, 3, 5, seed=2), MLP(7, hidden, 3, 5, seed=2)
    for m in (a, b):
        m.fit_normalization(x, t)
    p0 = a.params()
    loss, _ = a.train(x, t, epochs=steps, batch=n, lr=lr, seed=1)
    for _ in range(steps):
        last, _ = b.gradients(x, t)
        b.adam_step(lr)
    pa, pb = a.params(), b.params()
    moved = np.linalg.norm(pb - p0)
    assert moved > 0 and np.abs(pa - p0).max() <= 1.01 * steps * lr
    assert np.linalg.norm(pa - pb) <= 2e-2 * moved
    assert loss == pytest.approx(last, rel=1e-3)


def test_a_large_batch_keeps_its_gradients_chains_short():
    """The weight gradients of 2^19 samples whose targets are noise, against FP64 sums of the traced dZ
    and H: FP32 chains of c = 512 matrix products of 32 samples, then 32 partial sums. A chain of c
    zero-mean terms grows as the square root of its length and each addition rounds its value by 0.42
    2^-24 of it (the root mean square over a mantissa), so the chain ends 0.42 2^-24 sqrt(c / 2) of its
    value off, and the sum of 32 such adds 0.42 2^-24 sqrt(32 / 2): 4.2e-7 in all; eight partial sums
    would make it 8.1e-7."""
    n, u = 1 << 19, 0.424 * 2.0**-24
    x, _ = data(n, 7, 5, 3)
    t = np.random.default_rng(4).standard_normal((n, 5)).astype(np.float32)
    m = MLP(7, 64, 2, 5, seed=1)
    _, g = m.gradients(x, t)
    at = 0
    w = m.widths()
    for l in range(len(w) - 1):
        h, dz = m.trace(x, t, "input", l).astype(np.float64), m.trace(x, t, "dz", l).astype(np.float64)
        want = dz.T @ h
        got = g[at : at + want.size].reshape(want.shape)
        at += want.size + w[l + 1]
        assert np.linalg.norm(got - want) <= u * np.hypot(np.sqrt(512 / 2), np.sqrt(32 / 2)) * np.linalg.norm(want), l
    m.close()


def pair(hidden, x, t):
    a, b = MLP(7, hidden, 3, 5, seed=2), MLP(7, hidden, 3, 5, seed=2)
    for m in (a, b):
        m.fit_normalization(x, t)
    return a, b


@pytest.mark.parametrize("hidden,n", [(128, 500), (192, 500), (64, 8200), (128, 8193), (192, 8223), (256, 8200)])
def test_an_epoch_of_one_batch_at_every_width_and_tile(hidden, n):
    """As test_an_epoch_is_its_batches, to its bounds, at the other widths and past one row tile per
    workgroup."""
    steps, lr = 3, 1e-3
    x, t = data(n, 7, 5, 3)
    a, b = pair(hidden, x, t)
    p0 = a.params()
    loss, _ = a.train(x, t, epochs=steps, batch=n, lr=lr, seed=1)
    for _ in range(steps):
        last, _ = b.gradients(x, t)
        b.adam_step(lr)
    moved = np.linalg.norm(b.params() - p0)
    assert moved > 0 and np.linalg.norm(a.params() - b.params()) <= 2e-2 * moved
    assert loss == pytest.approx(last, rel=1e-3)


@pytest.mark.parametrize("hidden,batch", [(64, 100), (256, 256), (128, 8200)])
def test_every_batch_of_an_epoch_is_its_own(hidden, batch):
    """Four batches whose samples the shuffle chooses, at weights that stand still: the epoch's loss is
    the mean over its samples, here the count of those with a large target, 37 in all and at most the
    five samples left over fewer. A batch taken twice would make the count another, or by its size a
    multiple of four under every seed. With as many samples as the batches take, the loss is gradients()'s."""
    left, large = 5, 37
    n = 4 * batch + left
    x, _ = data(n, 7, 5, 3)
    t = np.zeros((n, 5), np.float32)
    t[np.random.default_rng(6).choice(n, large, replace=False)] = 1e4  # a large sample's squared error: 1e8, others' below 1
    m = MLP(7, hidden, 3, 5, seed=2)
    counts = []
    for seed in range(6):
        loss, _ = m.train(x, t, epochs=1, batch=batch, lr=0.0, seed=seed)
        count = loss * 4 * batch / 1e8
        assert abs(count - round(count)) <= 0.02 and large - left <= round(count) <= large, count
        counts.append(round(count))
    assert any(c % 4 for c in counts)
    whole = 4 * batch
    t[:, 0] += np.arange(n) ** 2  # targets unlike each other
    want, _ = m.gradients(x[:whole], t[:whole])
    loss, _ = m.train(x[:whole], t[:whole], epochs=1, batch=batch, lr=0.0, seed=7)
    # FP32 squared errors, summed to 64 lanes in FP32 and further in FP64, in another order
    assert loss == pytest.approx(want, rel=1e-5)
    m.close()


def test_steps_within_an_epoch_are_counted():
    """Batches all alike: an epoch of four is four of gradients() and adam_step(), whose bias corrections
    depend on the count."""
    one, lr = 128, 1e-3
    x, t = data(1, 7, 5, 3)
    x, t = np.tile(x, (4 * one, 1)), np.tile(t, (4 * one, 1))
    a, b = MLP(7, 128, 3, 5, seed=2), MLP(7, 128, 3, 5, seed=2)
    p0 = a.params()
    a.train(x, t, epochs=1, batch=one, lr=lr, seed=1)
    for _ in range(4):
        b.gradients(x[:one], t[:one])
        b.adam_step(lr)
    moved = np.linalg.norm(b.params() - p0)
    assert moved > 0 and np.linalg.norm(a.params() - b.params()) <= 1e-5 * moved


@pytest.mark.parametrize("hidden,layers", [(64, 2), (192, 3), (256, 2)])
@pytest.mark.parametrize("n", [17, 33, 8191, 8193, 8209])
def test_the_last_tile_alone(hidden, layers, n):
    """Targets of the last tile of 32 that are so large that its samples, one of 8193, are the gradient:
    a tile dropped, read twice or masked wrongly is all of it. To the bound of the tiles' edges test."""
    x, t = data(n, 7, 5, n)
    t[(n - 1) // 32 * 32 :] += 1e6
    m = MLP(7, hidden, layers, 5, seed=n)
    norm = [np.asarray(a, np.float64) for a in m.norm]
    loss, g = m.gradients(x, t)
    l_o, g_o = mo.loss_and_gradients(m.params(), m.widths(), x, t, norm, 5, bf=True)
    assert abs(loss - l_o) <= 1e-2 * l_o
    at = 0
    w = m.widths()
    for l in range(len(w) - 1):
        for size in (w[l + 1] * w[l], w[l + 1]):
            seg = slice(at, at + size)
            at += size
            assert np.linalg.norm(g[seg] - g_o[seg]) <= 5e-2 * np.linalg.norm(g_o[seg]), (l, size)
    m.close()
