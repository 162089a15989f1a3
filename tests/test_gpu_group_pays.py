"""Which gates an untimed sync takes in one pass: not a few that touch a small
part of a large state; and circuits of such gates against the oracle.

Relative L2 <= 1e-12 at f64 (a gate rounds at about 4 eps, 24 gates)."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
import oracle
from cast_simulator_amd import abi
from helpers import rel_l2
from test_gpu_groups import phase, unitary

pytestmark = pytest.mark.gpu


def toffoli(k):
    m = np.eye(1 << k, dtype=complex)
    a = (1 << k) - 1
    m[[a, a >> 1]] = m[[a >> 1, a]]
    return m


RNG = np.random.default_rng(1)
P = {k: phase(k, RNG) for k in range(1, 7)}


@pytest.mark.parametrize("gates,pays", [
    ([(P[2], [20, 21]), (P[2], [18, 19])], {20: True, 24: False, 30: False}),
    ([(P[5], [10, 12, 14, 16, 18]), (P[5], [11, 12, 14, 16, 18])], {20: True, 24: False, 30: False}),
    ([(P[2], [0, 1]), (P[2], [1, 2])], {20: True, 24: True, 30: True}),  # every line
    ([(P[2], [10 + i, 11 + i]) for i in range(6)], {20: True, 24: True, 30: True}),
    ([(toffoli(3), [15, 16, 18]), (toffoli(3), [14, 17, 19])], {20: True, 24: False, 30: False}),
    ([(unitary(1, RNG), [19]), (P[6], list(range(10, 16)))], {20: True, 24: True, 30: True}),
    ([(P[2], [20, 21])], {24: False}),
])
def test_rule(gates, pays):
    plans = [abi.plan_create(m, q, abi.F64) for m, q in gates]
    try:
        for n, want in pays.items():
            if max(max(q) for _, q in gates) < n:
                assert abi.gate_group_pays(plans, n) is want, n
    finally:
        for p in plans:
            abi.plan_destroy(p)


def test_sparse_circuit_matches_oracle():
    n = 23
    rng = np.random.default_rng(n)
    gates = []
    for i in range(24):
        k = 2 + int(rng.integers(4))
        q = sorted(rng.choice(n, k, replace=False).tolist())
        gates.append((unitary(2, rng), q[:2]) if i % 6 == 5 else
                     (P[k] if i % 2 else toffoli(k), q))
    x = np.asarray(cs.random_statevector(n, 1))
    mgr = cs.HipKernelManager(cs.HipKernelGenSpec.f64())
    sv = cs.HipStatevector(n, cs.Precision.F64)
    sv.upload(x)
    print(f"[group pays] n={n} sparse circuit", flush=True)
    for m, q in gates:
        mgr.apply(mgr.generate(cs.QuantumGate(m, q)), sv)
    mgr.sync(False)
    want = x.copy()
    oracle.apply_gates(want, gates)
    assert rel_l2(want, np.asarray(sv.download())) <= 1e-12
