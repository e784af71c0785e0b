"""Sums read back through pinned memory by the last workgroup to finish: one
workgroup and many, repeated, from several threads at once."""

import threading

import numpy as np
import pytest

import ember_amd as em
from ember_amd import loss
from ember_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [1, 255, 256, 257, 1000, 65536, 262143, 262145, 1 << 20, 5000003])
def test_sum_of_every_workgroup_count(size):
    x = np.random.default_rng(size).standard_normal(size, dtype=np.float32)
    t = Tensor(x)
    first = em.sum(t)
    # Doubles throughout and one rounding to fp32.
    exact = x.astype(np.float64).sum()
    assert first == pytest.approx(exact, rel=2.0 ** -23, abs=1e-9 * size)
    for _ in range(20):
        assert em.sum(t) == first


def test_threads_get_their_own_sums():
    rng = np.random.default_rng(0)
    xs = [Tensor(rng.standard_normal(n, dtype=np.float32)) for n in (3, 70000, 300000, 1500000)]
    logits = [Tensor(rng.standard_normal((n, 50), dtype=np.float32)) for n in (2, 700, 20000)]
    ts = [Tensor(np.full(x.shape, 0.02, np.float32)) for x in logits]
    want = [em.sum(x) for x in xs] + [loss.CrossEntropyLoss()(x, t) for x, t in zip(logits, ts)]
    bad = []

    def work():
        for _ in range(50):
            got = [em.sum(x) for x in xs] + [loss.CrossEntropyLoss()(x, t) for x, t in zip(logits, ts)]
            if got != want:
                bad.append(got)

    threads = [threading.Thread(target=work) for _ in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, (bad[0], want)
