"""The warm-start network's calls beside each other: predictions from several host threads at
once, what calls keep on the device, and data that does not fit there."""

from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from autan_amd.mlp import MLP
from hipmem import free_bytes

pytestmark = pytest.mark.gpu


def samples(n, seed):
    return np.random.default_rng(seed).uniform(-1, 1, size=(n, 7)).astype(np.float32)


def test_predictions_from_several_threads():
    """Each call has its own device copies of its samples, so calls of unlike sizes at the same time
    return what they return alone, bit for bit."""
    m = MLP(7, 128, 3, 5, seed=4)
    xs = [samples(n, n) for n in (1, 700, 5000, 90000)]
    want = [m.predict(x) for x in xs]
    wrong = []

    def calls(k):
        for _ in range(20):
            if not np.array_equal(m.predict(xs[k]), want[k]):
                wrong.append(xs[k].shape[0])

    threads = [threading.Thread(target=calls, args=(k,)) for k in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    m.close()


@pytest.mark.parametrize("hidden,fused", [(320, True), (256, False)])
def test_layered_prediction_holds_a_chunk_of_activations(hidden, fused):
    """Layer by layer a prediction of many samples goes by chunks of 2^16, whose activations (BF16),
    pre-activations (FP32) and gradients' room (BF16) of every layer stay on the device: 8 bytes per
    value of a layer."""
    m = MLP(7, hidden, 3, 5, seed=4)
    m.set_fused(fused)
    x = samples((1 << 18) + 3, 8)
    m.predict(x[:64])
    before = free_bytes()
    y = m.predict(x)
    grown = before - free_bytes()
    held = (1 << 16) * (8 * sum(m.widths()[1:]) + 2 * 32)
    assert grown <= held + (64 << 20)  # the chunk's samples and the allocator's granularity
    np.testing.assert_array_equal(m.predict(x[-5000:]), y[-5000:])
    m.close()


def test_a_wide_network_holds_no_operand_packs():
    """Networks wider than the fused kernels hold, per parameter, the FP32 weight, gradient and Adam's
    two moments, the BF16 weight and a mask byte: nothing laid out for kernels that they never run."""
    small = MLP(7, 64, 1, 5)  # what a process's first network makes the runtime allocate
    small.predict(samples(10, 1))
    before = free_bytes()
    m = MLP(7, 2048, 4, 5, seed=4)
    assert before - free_bytes() <= m.param_count * (4 * 4 + 2 + 1) + (32 << 20)
    m.close()
    small.close()


def test_data_that_does_not_fit_leaves_none():
    """Training data whose inputs fit the device (34 GB) and whose targets do not (550 GB): the call is
    refused before it reads a sample, and training is until there is data again."""
    m = MLP(1, 64, 1, 16, seed=1)
    x, t = samples(64, 1)[:, :1].copy(), np.zeros((64, 16), np.float32)
    loss, _ = m.train(x, t, epochs=1, batch=64, lr=0.0)
    with pytest.raises(RuntimeError, match="hipMalloc"):
        m._call(m.lib.mxmlp_set_data, ctypes.c_void_p(x.ctypes.data), ctypes.c_void_p(t.ctypes.data),
                ctypes.c_int64(1 << 33))
    out, sec = ctypes.c_float(), ctypes.c_double()
    with pytest.raises(RuntimeError, match="batch >= 64 and <= the data"):
        m._call(m.lib.mxmlp_train, ctypes.c_int32(1), ctypes.c_int32(64), ctypes.c_float(0.0), ctypes.c_uint64(0),
                ctypes.byref(out), ctypes.byref(sec))
    assert m.train(x, t, epochs=1, batch=64, lr=0.0)[0] == pytest.approx(loss, rel=1e-6)
    m.close()
