"""Amplitudes that a monomial gate does not touch stay as they are in a group,
infinities among them, as in a launch of the gate by itself."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
from cast_simulator_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
@pytest.mark.parametrize("k", [2, 4])
def test_identity_rows_of_permutations_keep_infinities(precision, k):
    """k = 4 at f64 is wider than the thread's registers."""
    n = 10
    m = np.eye(1 << k, dtype=complex)
    m[[1, 2]] = m[[2, 1]] * np.exp(0.3j)
    q = [0, 3, 7, 9][:k]
    x = np.asarray(cs.random_statevector(n, 4))
    idx = np.arange(1 << n)
    row = sum(((idx >> p) & 1) << b for b, p in enumerate(q))
    x[2 * idx[row == 0][5]] = np.inf
    x[2 * idx[row == 3][7] + 1] = -np.inf
    want = x.astype(np.float32).astype(np.float64) if precision == abi.F32 else x
    plan = abi.plan_create(m, q, precision)
    sv = abi.sv_alloc(n, precision)
    got = []
    try:
        print(f"[group infinite] precision={precision} k={k}", flush=True)
        for launch in (abi.gate_apply, lambda p, s, n: abi.gate_apply_group([p], s, n)):
            abi.sv_upload(sv, x, precision)
            launch(plan, sv, n)
            abi.stream_sync(None)
            got.append(np.asarray(abi.sv_download(sv, n, precision)).reshape(-1, 2))
    finally:
        abi.sv_free(sv)
        abi.plan_destroy(plan)
    kept = (row != 1) & (row != 2)
    for g in got:
        np.testing.assert_array_equal(g[kept], want.reshape(-1, 2)[kept])
        assert np.isfinite(g[~kept]).all()


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
@pytest.mark.parametrize("k", [3, 4, 5, 6])
def test_identity_entries_of_diagonals_keep_infinities(precision, k):
    n = 10
    rows = np.arange(1 << k)
    phased = rows % 3 == 1
    m = np.diag(np.where(phased, np.exp(0.1j * rows), 1.0))
    q = [0, 2, 3, 5, 7, 9][:k]
    x = np.asarray(cs.random_statevector(n, 6))
    idx = np.arange(1 << n)
    row = sum(((idx >> p) & 1) << b for b, p in enumerate(q))
    for r in rows[~phased]:
        x[2 * idx[row == r][3] + r % 2] = np.inf
    want = x.astype(np.float32).astype(np.float64) if precision == abi.F32 else x
    plan = abi.plan_create(m, q, precision)
    sv = abi.sv_alloc(n, precision)
    try:
        print(f"[group infinite] diagonal precision={precision} k={k}", flush=True)
        abi.sv_upload(sv, x, precision)
        abi.gate_apply_group([plan], sv, n)
        abi.stream_sync(None)
        got = np.asarray(abi.sv_download(sv, n, precision)).reshape(-1, 2)
    finally:
        abi.sv_free(sv)
        abi.plan_destroy(plan)
    kept = ~phased[row]
    np.testing.assert_array_equal(got[kept], want.reshape(-1, 2)[kept])
    amp = (want.reshape(-1, 2)[~kept] @ [1, 1j]) * np.exp(0.1j * row[~kept])
    tol = 8 * (np.finfo(np.float32).eps if precision == abi.F32 else np.finfo(np.float64).eps)
    np.testing.assert_allclose(got[~kept] @ [1, 1j], amp, rtol=tol, atol=0)
