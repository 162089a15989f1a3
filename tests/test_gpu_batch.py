"""Batched gates where the batch changes kernel: matrix cores from k + 4 qubits
on, the direct kernel below, in one call, against the oracle.

Tolerances as for single gates: relative L2 <= 1e-13 at f64 (one gate of K <=
64 terms rounds below 1e-14) and <= 1e-6 at f32 (a gate rounds at about 2e-7)."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
import oracle
from cast_simulator_amd import abi
from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [(abi.F64, 1e-13), (abi.F32, 1e-6)])
@pytest.mark.parametrize("k", [4, 5, 6])
def test_batch_of_mixed_sizes_matches_oracle(k, precision, tol):
    rng = np.random.default_rng(10 * k + precision)
    sizes = [k, k + 3, k + 4, k + 5, 12, 15, k + 4, 13] * 9  # more than one launch
    items = []
    for i, n in enumerate(sizes):
        m = rng.standard_normal((1 << k, 1 << k)) + 1j * rng.standard_normal((1 << k, 1 << k))
        m = np.linalg.qr(m)[0]
        if i % 7 == 3:
            m = np.diag(np.exp(2j * np.pi * rng.random(1 << k)))  # monomial
        q = sorted(rng.choice(n, k, replace=False).tolist())
        x = np.asarray(cs.random_statevector(n, 500 + i))
        sv = abi.sv_alloc(n, precision)
        abi.sv_upload(sv, x, precision)
        items.append((n, m, q, x, sv, abi.plan_create(m, q, precision)))
    try:
        abi.gate_apply_batch([t[5] for t in items], [t[4] for t in items], [t[0] for t in items])
        abi.stream_sync(None)
        for n, m, q, x, sv, _ in items:
            want = x.astype(np.float32) if precision == abi.F32 else x.copy()
            oracle.apply_gates(want, [(m, q)])
            assert rel_l2(want.astype(np.float64), abi.sv_download(sv, n, precision)) <= tol, (n, q)
    finally:
        for t in items:
            abi.sv_free(t[4])
            abi.plan_destroy(t[5])
