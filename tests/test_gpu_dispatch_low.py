"""Single gates where targets crowd in the lowest bits or the state fits the XCDs'
L2, and diagonal gates on both sides of the share of lines at which
they go as a stream: the kernel chosen, and the result against the oracle.

Relative L2 <= 1e-13 at f64 (one gate of K <= 64 terms rounds below 1e-14) and
<= 1e-6 at f32 (a gate rounds at about 2e-7)."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
from cast_simulator_amd import abi
from test_gpu_dispatch import TOL, apply_one
from test_gpu_groups import unitary

pytestmark = pytest.mark.gpu

DIRECT, TILE, CORES = 1, 3, 4


@pytest.mark.parametrize("precision,n,q,family", [
    (abi.F64, 22, [0, 1], TILE), (abi.F64, 22, [0, 2], DIRECT), (abi.F64, 22, [0, 1, 9], TILE),
    (abi.F64, 22, [1, 2, 9], DIRECT), (abi.F64, 20, [5], TILE), (abi.F64, 20, [18, 19], TILE),
    (abi.F64, 20, [2, 3, 4], TILE), (abi.F64, 20, [0, 7, 8, 9], TILE),
    (abi.F64, 20, [0, 1, 2, 3], CORES), (abi.F64, 19, [18], TILE), (abi.F64, 21, [9, 10], DIRECT),
    (abi.F64, 18, [0, 1], TILE), (abi.F64, 18, [0, 1, 2], DIRECT),
    (abi.F64, 21, [7, 8, 9, 10, 11], CORES), (abi.F64, 22, [7, 8, 9, 10, 11], TILE),
    (abi.F32, 22, [0, 2], TILE), (abi.F32, 22, [0, 3], DIRECT), (abi.F32, 22, [0, 1, 2], TILE),
    (abi.F32, 22, [0, 1, 3], DIRECT), (abi.F32, 21, [20], TILE), (abi.F32, 20, [4, 9, 11], TILE),
    (abi.F32, 20, [4, 9, 11, 13], TILE), (abi.F32, 19, [4, 9, 11], DIRECT),
    (abi.F32, 23, [0, 1, 2, 9], CORES), (abi.F32, 23, [0, 1, 3, 9], DIRECT),
    (abi.F32, 24, [20, 21, 22, 23], DIRECT), (abi.F32, 23, [19, 20, 21, 22], TILE),
])
def test_chosen_kernel(precision, n, q, family):
    rng = np.random.default_rng(n + len(q))
    m = unitary(len(q), rng)
    plan = abi.plan_create(m, q, precision)
    try:
        assert abi.plan_family(plan, n) == family
    finally:
        abi.plan_destroy(plan)
    if n <= 22:  # the kernels are the same above
        assert apply_one(m, q, n, precision, np.asarray(cs.random_statevector(n, n))) <= TOL[precision]


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
@pytest.mark.parametrize("n", [20, 22])
def test_diagonals_around_the_share_of_a_stream(n, precision):
    rng = np.random.default_rng(n)
    x = np.asarray(cs.random_statevector(n, n))
    for k in (2, 3, 4, 5):
        K = 1 << k
        for ones in (0, 1, K // 8, K // 4):
            d = np.exp(2j * np.pi * rng.random(K))
            d[:ones] = 1.0
            for q in (list(range(n - k, n)), [1] + list(range(n - k + 1, n))):
                err = apply_one(np.diag(d), q, n, precision, x)
                assert err <= TOL[precision], (k, ones, q, err)
