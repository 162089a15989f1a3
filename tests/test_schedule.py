"""Cutting gate lists into passes (host only): every gate runs once, gates that
share a qubit keep their order, and a pass keeps to its limits."""
from __future__ import annotations

import numpy as np
import pytest

from cast_simulator_amd import _host


@pytest.mark.parametrize("n,max_qubits,low,max_gates", [
    (30, 12, 4, 64), (30, 13, 4, 64), (16, 12, 4, 5), (12, 12, 4, 64), (34, 13, 4, 64),
])
@pytest.mark.parametrize("seed", [1, 2, 3])
def test_passes_keep_order_and_limits(n, max_qubits, low, max_gates, seed):
    rng = np.random.default_rng(seed)
    gates = [sorted(rng.choice(n, int(rng.integers(1, 7)), replace=False).tolist())
             for _ in range(120)]
    joins = [len(q) <= 5 and rng.random() < 0.9 for q in gates]
    passes = _host.plan_passes(gates, joins, n, max_qubits, low, max_gates)
    order = [i for p in passes for i in p]
    assert sorted(order) == list(range(len(gates)))
    at = {g: i for i, g in enumerate(order)}
    for i in range(len(gates)):
        for j in range(i):
            if set(gates[i]) & set(gates[j]):
                assert at[j] < at[i]
    for p in passes:
        assert p == sorted(p) and 1 <= len(p) <= max_gates
        if len(p) > 1:
            assert all(joins[i] for i in p)
            assert len(set(range(low)).union(*(gates[i] for i in p))) <= max_qubits
    assert len(passes) < len(gates)


def test_no_gates():
    assert _host.plan_passes([], [], 20, 12, 4, 64) == []
