"""Gate groups on statevectors that fill the chip (from 22 qubits f64, 23 f32),
where a thread holds twice the amplitudes and tiles go in XCD order, against
the oracle: every kind and size of gate with targets at both edges of the tile,
and untimed circuits over the whole statevector.

Tolerances as for the smaller groups: relative L2 <= 1e-12 at f64 (a gate
rounds at about K eps < 1e-14, and a case has at most 64 gates) and <= 1e-5 at
f32 (a gate rounds at about 2e-7, and a case has at most 40)."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
import oracle
from cast_simulator_amd import abi
from helpers import rel_l2
from test_gpu_groups import TOL, diagonal, permutation, phase, run_group, target_sets, unitary

pytestmark = pytest.mark.gpu

LARGE = {abi.F64: 22, abi.F32: 23}


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
@pytest.mark.parametrize("kind,top", [(unitary, 5), (permutation, 4), (diagonal, 6), (phase, 6)])
def test_every_kind_on_a_full_chip(precision, kind, top):
    n = LARGE[precision]
    rng = np.random.default_rng(n + precision)
    low, room = (2, 12) if precision == abi.F64 else (3, 13)
    # a tile of low and high qubits that leaves the ones between out
    pool = list(range(low)) + list(range(n - (room - low), n))
    gates = [(unitary(1, rng), [q]) for q in pool[::4]]
    for k in range(1, top + (kind is unitary and precision == abi.F32) + 1):
        gates += [(kind(k, rng), q) for q in target_sets(k, pool)]
    print(f"[group large] n={n} precision={precision} {kind.__name__} {len(gates)} gates", flush=True)
    assert run_group(gates, n, precision, 3 * n) <= TOL[precision]


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
def test_untimed_mixed_circuit_on_a_full_chip(precision):
    n, f32 = LARGE[precision], precision == abi.F32
    rng = np.random.default_rng(9 + precision)
    gates = []
    for i in range(36):
        kind = [unitary, unitary, permutation, diagonal, phase][i % 5]
        k = 1 + int(rng.integers(4 if kind is permutation else 6))
        gates.append((kind(k, rng), sorted(rng.choice(n, k, replace=False).tolist())))
    x = np.asarray(cs.random_statevector(n, n))
    mgr = cs.HipKernelManager(cs.HipKernelGenSpec.f32() if f32 else cs.HipKernelGenSpec.f64())
    sv = cs.HipStatevector(n, cs.Precision.F32 if f32 else cs.Precision.F64)
    sv.upload(x)
    print(f"[group large] n={n} precision={precision} mixed circuit", flush=True)
    for m, q in gates:
        mgr.apply(mgr.generate(cs.QuantumGate(m, q)), sv)
    mgr.sync(False)
    want = x.astype(np.float32) if f32 else x.copy()
    oracle.apply_gates(want, gates)
    assert rel_l2(want.astype(np.float64), np.asarray(sv.download())) <= TOL[precision]
