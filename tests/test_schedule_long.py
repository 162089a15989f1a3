"""Long gate lists (host only): planning takes about as long per gate where a
qubit is idle as where none is, and no gate is lost or moved past another that
shares a qubit."""
from __future__ import annotations

import time

import numpy as np
import pytest

from cast_simulator_amd import _host


def random_pairs(n_used, count, seed):
    rng = np.random.default_rng(seed)
    a = rng.integers(n_used, size=count)
    b = (a + 1 + rng.integers(n_used - 1, size=count)) % n_used
    return [sorted(p) for p in zip(a.tolist(), b.tolist())]


def seconds(n_used, count):
    gates = random_pairs(n_used, count, 1)
    best = 1e9
    for _ in range(3):
        t = time.perf_counter()
        _host.plan_passes(gates, [True] * count, 20, 12, 2, 64)
        best = min(best, time.perf_counter() - t)
    return best


def test_idle_qubit_does_not_slow_planning():
    """Looking through the whole list for every pass takes 20 times as long."""
    assert seconds(19, 16000) <= 8 * seconds(20, 16000)


@pytest.mark.parametrize("n_used,joins", [(19, 1.0), (20, 1.0), (18, 0.9), (5, 1.0), (20, 0.0)])
def test_long_lists_keep_order(n_used, joins):
    gates = random_pairs(n_used, 2500, n_used)
    may = (np.random.default_rng(3).random(len(gates)) < joins).tolist()
    passes = _host.plan_passes(gates, may, 20, 12, 2, 64)
    order = [i for p in passes for i in p]
    assert sorted(order) == list(range(len(gates)))
    last = {}
    for i in order:  # ascending on every qubit
        for q in gates[i]:
            assert last.get(q, -1) < i
            last[q] = i
    for p in passes:
        assert p == sorted(p) and len(p) <= 64
        if len(p) > 1:
            assert all(may[i] for i in p)
            assert len({0, 1}.union(*(gates[i] for i in p))) <= 12
