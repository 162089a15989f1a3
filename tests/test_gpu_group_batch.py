"""Groups on several statevectors in shared launches: the same bits as one
launch per group, and members of an ensemble against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
import oracle
from cast_simulator_amd import abi
from helpers import rel_l2
from test_gpu_groups import TOL, diagonal, permutation, phase, unitary

pytestmark = pytest.mark.gpu


def random_groups(rng, n, precision, states, rounds):
    """Per state a list of groups of every kind of gate within one tile."""
    room = min(n, 12 if precision == abi.F64 else 13)
    kinds = [(unitary, 6 if precision == abi.F64 else 7), (permutation, 5), (diagonal, 7), (phase, 7)]
    out = []
    for s in range(states):
        groups = []
        for _ in range(1 + (s + rounds) % (rounds + 1)):
            pool = list(range(3)) + sorted(rng.choice(np.arange(3, n), room - 3, replace=False).tolist())
            gates = []
            for _ in range(int(rng.integers(1, 8))):
                kind, top = kinds[int(rng.integers(4))]
                k = int(rng.integers(1, top))
                gates.append((kind(k, rng), sorted(rng.choice(pool, k, replace=False).tolist())))
            groups.append(gates)
        out.append(groups)
    return out


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
@pytest.mark.parametrize("n,states", [(10, 1), (11, 3), (13, 17), (17, 5), (21, 2)])
def test_shared_launches_equal_single_ones(precision, n, states):
    rng = np.random.default_rng(10 * n + precision)
    dt = np.float64 if precision == abi.F64 else np.float32
    work = random_groups(rng, n, precision, states, 3)
    plans = [[[abi.plan_create(m, q, precision) for m, q in g] for g in groups] for groups in work]
    svs = [[abi.malloc((2 << n) * dt().itemsize) for _ in range(states)] for _ in range(2)]
    n_groups = sum(len(p) for p in plans)
    scratch = abi.malloc(abi.group_batch_scratch_bytes(n_groups, sum(len(g) for p in plans for g in p)))
    print(f"[group batch] n={n} precision={precision} states={states} groups={n_groups}", flush=True)
    try:
        for s in range(states):
            x = rng.standard_normal(2 << n).astype(dt)
            for side in svs:
                abi.memcpy_htod(side[s], x)
            for g in plans[s]:
                abi.gate_apply_group(g, svs[0][s], n)
        items = [(plans[s][r], svs[1][s], r) for r in range(4) for s in range(states)
                 if r < len(plans[s])]
        abi.gate_apply_group_batch(items, n, scratch)
        abi.stream_sync(None)
        for s in range(states):
            a, b = np.zeros(2 << n, dt), np.zeros(2 << n, dt)
            abi.memcpy_dtoh(a, svs[0][s])
            abi.memcpy_dtoh(b, svs[1][s])
            np.testing.assert_array_equal(a, b)
    finally:
        for p in svs[0] + svs[1] + [scratch]:
            abi.free(p)
        for p in plans:
            for g in p:
                for h in g:
                    abi.plan_destroy(h)


def test_refused_calls():
    h = abi.plan_create(unitary(1, np.random.default_rng(0)), [0], abi.F64)
    sv = abi.malloc(16 << 10)
    try:
        with pytest.raises(abi.AbiError, match="must not decrease"):
            abi.gate_apply_group_batch([([h], sv, 1), ([h], sv, 0)], 10, sv)
        with pytest.raises(abi.AbiError, match="fill the chip"):
            abi.gate_apply_group_batch([([h], sv, 0)], 22, sv)
        with pytest.raises(abi.AbiError, match="no plans"):
            abi.gate_apply_group_batch([([], sv, 0)], 10, sv)
        with pytest.raises(abi.AbiError, match="scratch"):
            abi.gate_apply_group_batch([([h], sv, 0)], 10, 0)
    finally:
        abi.free(sv)
        abi.plan_destroy(h)


@pytest.mark.parametrize("n", [8, 10, 13])
@pytest.mark.parametrize("f32", [False, True])
def test_many_statevectors_of_one_manager(n, f32):
    """Untimed work on statevectors with different gate lists, some of one gate."""
    rng = np.random.default_rng(n)
    prec = cs.Precision.F32 if f32 else cs.Precision.F64
    mgr = cs.HipKernelManager(cs.HipKernelGenSpec.f32() if f32 else cs.HipKernelGenSpec.f64())
    svs, want = [], []
    for s in range(5):
        x = np.asarray(cs.random_statevector(n, s))
        sv = cs.HipStatevector(n, prec)
        sv.upload(list(x))
        w = x.astype(np.float32) if f32 else x.copy()
        for _ in range([1, 7, 12, 1, 20][s]):
            k = int(rng.integers(1, 7))
            m, q = unitary(k, rng), sorted(rng.choice(n, k, replace=False).tolist())
            mgr.apply(mgr.generate(cs.QuantumGate(m, q)), sv)
            oracle.apply_gate(w, m, q)
        svs.append(sv)
        want.append(w)
    mgr.sync(False)
    for sv, w in zip(svs, want):
        assert rel_l2(w.astype(np.float64), np.asarray(sv.download())) <= TOL[0 if f32 else 1]
