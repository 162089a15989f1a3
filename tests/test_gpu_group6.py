"""Six-qubit f32 gates in groups (split products with streamed operands)
against the oracle; bounds and helpers are those of the other groups."""
from __future__ import annotations

import numpy as np
import pytest

from cast_simulator_amd import abi
from test_gpu_groups import TOL, phase, run_group, target_sets, unitary

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [10, 11, 13, 14, 16, 23])
def test_group_with_six_qubit_gates(n):
    """One wave and one tile of combos (n = 10) up to two tiles a wave (n = 23)."""
    rng = np.random.default_rng(n)
    pool = list(range(3)) + list(range(n - min(n, 13) + 3, n))
    gates = [(unitary(6, rng), q) for q in target_sets(6, pool)]
    gates += [(unitary(5, rng), pool[-5:]), (phase(6, rng), pool[1:7]), (unitary(3, rng), pool[:3])]
    gates.append((unitary(6, rng), sorted(rng.choice(pool, 6, replace=False).tolist())))
    assert run_group(gates, n, abi.F32, n) <= TOL[abi.F32]


def test_double_precision_stays_alone():
    """f64 k = 6 keeps its own pass."""
    m = unitary(6, np.random.default_rng(0))
    for precision, joins in ((abi.F32, True), (abi.F64, False)):
        p = abi.plan_create(m, list(range(6)), precision)
        assert bool(abi.gate_group_info(p, 20).targets) is joins
        abi.plan_destroy(p)
