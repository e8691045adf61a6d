"""The warm-start network's calls beside each other: predictions from several host threads at once."""

from __future__ import annotations

import threading

import numpy as np
import pytest

from autan_amd.mlp import MLP

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
