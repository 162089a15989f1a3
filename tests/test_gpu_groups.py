"""Gate groups (several gates in one pass over the statevector) against the
oracle: every kind of gate, at the smallest and largest tiles, with targets at
the edges of the tile; and untimed circuits through the kernel manager.

Tolerances as in the single-gate tests: relative L2 <= 1e-12 at f64 (a gate
rounds at about K eps < 1e-14, and a case has at most 64 gates) and <= 1e-5 at
f32 (a gate rounds at about 2e-7, and a case has at most 40)."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
import oracle
from cast_simulator_amd import abi
from helpers import gate_list, rel_l2

pytestmark = pytest.mark.gpu

TOL = {abi.F64: 1e-12, abi.F32: 1e-5}


def unitary(k, rng):
    z = rng.standard_normal((1 << k, 1 << k)) + 1j * rng.standard_normal((1 << k, 1 << k))
    return np.linalg.qr(z)[0]


def permutation(k, rng):
    m = np.zeros((1 << k, 1 << k), dtype=complex)
    m[np.arange(1 << k), rng.permutation(1 << k)] = np.exp(2j * np.pi * rng.random(1 << k))
    return m


def diagonal(k, rng):
    d = np.exp(2j * np.pi * rng.random(1 << k))
    d[rng.random(1 << k) < 0.3] = 1.0
    return np.diag(d)


def phase(k, rng):
    return np.diag([1.0] * ((1 << k) - 1) + [np.exp(0.3j)])


def run_group(gates, n, precision, seed):
    """The gates as one group, and by the oracle."""
    init = np.asarray(cs.random_statevector(n, seed))
    plans = [abi.plan_create(m, q, precision) for m, q in gates]
    sv = abi.sv_alloc(n, precision)
    try:
        abi.sv_upload(sv, init, precision)
        abi.gate_apply_group(plans, sv, n)
        abi.stream_sync(None)
        got = abi.sv_download(sv, n, precision)
    finally:
        abi.sv_free(sv)
        for p in plans:
            abi.plan_destroy(p)
    want = init.astype(np.float32) if precision == abi.F32 else init.copy()
    oracle.apply_gates(want, gates)
    return rel_l2(want.astype(np.float64), got)


def target_sets(k, pool):
    """The lowest, the highest and a spread choice of k qubits of the pool."""
    step = max(1, (len(pool) - 1) // max(1, k - 1)) if k > 1 else 1
    sets = {tuple(pool[:k]), tuple(pool[-k:]), tuple(pool[:: step][:k])}
    return [list(s) for s in sorted(sets) if len(s) == k]


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
@pytest.mark.parametrize("kind,ks", [(unitary, range(1, 6)), (permutation, range(1, 5)),
                                     (diagonal, range(1, 7)), (phase, range(1, 7))])
@pytest.mark.parametrize("extra", [0, 1, 2, 3, 5])
def test_group_of_every_kind(precision, kind, ks, extra):
    n = (10 if precision == abi.F64 else 11) + extra
    rng = np.random.default_rng(100 * n + precision)
    room = min(n, 12 if precision == abi.F64 else 13)
    # a tile that skips qubits where the statevector has more than it holds
    low = 2 if precision == abi.F64 else 3
    pool = list(range(low)) + list(range(n - (room - low), n))
    for k in ks:
        gates = [(kind(k, rng), q) for q in target_sets(k, pool)]
        gates += [(unitary(1, rng), [q]) for q in pool]
        err = run_group(gates, n, precision, 7 + k)
        assert err <= TOL[precision], (kind.__name__, k, n, err)


@pytest.mark.parametrize("precision,n", [(abi.F64, 10), (abi.F64, 16), (abi.F32, 11),
                                         (abi.F32, 17)])
def test_group_of_mixed_gates(precision, n):
    rng = np.random.default_rng(n)
    pool = list(range(4)) + sorted(rng.choice(np.arange(4, n), min(n, 12) - 4, replace=False).tolist())
    gates = []
    for _ in range(40):
        kind = [unitary, unitary, permutation, diagonal, phase][int(rng.integers(5))]
        k = int(rng.integers(1, 5 if kind is permutation else 6))
        gates.append((kind(k, rng), sorted(rng.choice(pool, k, replace=False).tolist())))
    assert run_group(gates, n, precision, n) <= TOL[precision]


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,k", [(9, 3), (10, 2), (11, 4), (12, 5), (13, 6), (15, 3), (17, 5)])
def test_untimed_circuit_matches_oracle(n, k, f32):
    graph = cs.CircuitGraph.from_circuit(cs.random_layer_circuit(n, 6, 40 + n))
    cs.optimize(graph, cs.FusionConfig.size_only(k))
    gates = graph.gates_in_row_order()
    init = np.asarray(cs.random_statevector(n, n))
    mgr = cs.HipKernelManager(cs.HipKernelGenSpec.f32() if f32 else cs.HipKernelGenSpec.f64())
    two = [cs.HipStatevector(n, cs.Precision.F32 if f32 else cs.Precision.F64) for _ in range(2)]
    for sv in two:
        sv.upload(init)
    for g in gates:  # two statevectors in one queue
        for sv in two:
            mgr.apply(mgr.generate(g), sv)
    kernels, _ = mgr.sync(False)
    assert kernels == []
    want = init.astype(np.float32) if f32 else init.copy()
    oracle.apply_gates(want, gate_list(gates))
    for sv in two:
        assert rel_l2(want.astype(np.float64), np.asarray(sv.download())) <= TOL[0 if f32 else 1]


def test_group_limits_are_checked():
    rng = np.random.default_rng(1)
    n = 16
    far = [abi.plan_create(unitary(4, rng), [4 * i, 4 * i + 1, 4 * i + 2, 4 * i + 3], abi.F64)
           for i in range(4)]
    big = abi.plan_create(unitary(6, rng), [0, 1, 2, 3, 4, 5], abi.F64)
    single = abi.plan_create(unitary(1, rng), [0], abi.F32)
    sv = abi.sv_alloc(n, abi.F64)
    try:
        assert abi.gate_group_info(big, n).targets == 0
        assert abi.gate_group_info(far[3], n).targets == 0xF000
        assert abi.gate_group_info(far[3], 12).targets == 0
        with pytest.raises(abi.AbiError, match="more than 12 qubits"):
            abi.gate_apply_group(far, sv, n)
        with pytest.raises(abi.AbiError, match="cannot join"):
            abi.gate_apply_group([far[0], big], sv, n)
        with pytest.raises(abi.AbiError, match="share the precision"):
            abi.gate_apply_group([far[0], single], sv, n)
        with pytest.raises(abi.AbiError, match="at most"):
            abi.gate_apply_group([far[0]] * 65, sv, n)
    finally:
        abi.sv_free(sv)
        for p in far + [big, single]:
            abi.plan_destroy(p)
