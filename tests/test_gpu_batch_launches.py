"""The count of launches of a batch: 64 items a launch, items on the matrix
cores and on the direct kernel apart."""
from __future__ import annotations

import numpy as np
import pytest

from cast_simulator_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("direct,cores,launches", [
    (0, 0, 0), (1, 0, 1), (0, 64, 1), (0, 65, 2), (1, 1, 2), (64, 64, 2), (65, 63, 3), (3, 130, 4),
])
def test_launches_of_a_batch(direct, cores, launches):
    k = 5
    rng = np.random.default_rng(0)
    m = np.linalg.qr(rng.standard_normal((32, 32)) + 1j * rng.standard_normal((32, 32)))[0]
    dense = abi.plan_create(m, list(range(k)), abi.F64)
    diagonal = abi.plan_create(np.diag(np.exp(1j * np.arange(32.0))), list(range(k)), abi.F64)
    try:
        plans, sizes = [dense] * cores, [k + 4 + i % 3 for i in range(cores)]
        for i in range(direct):  # too small, or monomial
            plans.append(dense if i % 2 else diagonal)
            sizes.append(k + 3 if i % 2 else 14)
        assert abi.gate_batch_launches(plans, sizes) == launches
    finally:
        abi.plan_destroy(dense)
        abi.plan_destroy(diagonal)
