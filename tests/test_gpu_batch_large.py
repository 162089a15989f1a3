"""Batched f64 gates on both sides of 18 qubits, where k = 4, 5 go back to the
direct kernel unless targets crowd in the lowest bits: bit for bit the direct
kernel there, and the oracle's result everywhere (relative L2 <= 1e-13, one gate
of K <= 64 terms rounds below 1e-14)."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
import oracle
from cast_simulator_amd import abi
from helpers import rel_l2
from test_gpu_groups import unitary

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [4, 5, 6])
@pytest.mark.parametrize("n", [18, 19, 21])
def test_batch_around_eighteen_qubits(k, n):
    rng = np.random.default_rng(n + k)
    x = np.asarray(cs.random_statevector(n, n))
    for q in (list(range(k)), list(range(n - k, n)), [0] + list(range(5, 4 + k))):
        m = unitary(k, rng)
        plans = [abi.plan_create(m, q, abi.F64), abi.plan_create(m, q, abi.F64, variant=abi.VARIANT_DENSE)]
        svs = [abi.sv_alloc(n, abi.F64) for _ in range(3)]
        got = []
        try:
            for sv in svs:
                abi.sv_upload(sv, x, abi.F64)
            cores = k == 6 or n <= 18 or q[k - 3] < 3
            assert abi.gate_batch_launches(plans, [n, n]) == 1 + cores
            abi.gate_apply_batch([plans[0], plans[0], plans[1]], svs, [n] * 3)
            abi.stream_sync(None)
            got = [np.asarray(abi.sv_download(sv, n, abi.F64)) for sv in svs]
        finally:
            for sv in svs:
                abi.sv_free(sv)
            for p in plans:
                abi.plan_destroy(p)
        want = x.copy()
        oracle.apply_gates(want, [(m, q)])
        assert rel_l2(want, got[0]) <= 1e-13
        np.testing.assert_array_equal(got[0], got[1])
        if not cores:
            np.testing.assert_array_equal(got[0], got[2])
