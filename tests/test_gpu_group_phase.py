"""Diagonal gates with one entry other than 1, at every row, in groups against
the oracle (bounds and helpers of the other groups)."""
from __future__ import annotations

import numpy as np
import pytest

from cast_simulator_amd import abi
from test_gpu_groups import TOL, run_group, target_sets, unitary

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
@pytest.mark.parametrize("n", [10, 12, 16, 23])
def test_phase_at_every_row(precision, n):
    rng = np.random.default_rng(n + precision)
    room = min(n, 12 if precision == abi.F64 else 13)
    pool = list(range(3)) + list(range(n - room + 3, n))
    gates = [(unitary(1, rng), [q]) for q in pool]
    for k in range(1, 7):
        for q in target_sets(k, pool):
            d = np.ones(1 << k, complex)
            d[int(rng.integers(1 << k))] = [np.exp(1j * rng.uniform(0, 6)), -1, 0.5j][int(rng.integers(3))]
            gates.append((np.diag(d), q))
    assert len(gates) <= 40
    assert run_group(gates, n, precision, n) <= TOL[precision]


@pytest.mark.parametrize("k", [1, 2, 3, 4, 6])
def test_untouched_rows_keep_their_bits(k):
    """Infinities, NaN and signed zeros outside the row stay as they are."""
    n, row = 12, (1 << k) - 2 if k > 1 else 1
    rng = np.random.default_rng(k)
    q = sorted(rng.choice(n, k, replace=False).tolist())
    x = rng.standard_normal((1 << n, 2))
    at = np.zeros(1 << n, int)
    for b, t in enumerate(q):
        at |= ((np.arange(1 << n) >> t) & 1) << b
    rest = np.flatnonzero(at != row)
    x[rest[:4]] = [[np.inf, -0.0], [np.nan, 1.0], [-0.0, 0.0], [-np.inf, np.inf]]
    d = np.ones(1 << k, complex)
    d[row] = 1j
    plan = abi.plan_create(np.diag(d), q, abi.F64)
    sv = abi.malloc(x.nbytes)
    try:
        abi.memcpy_htod(sv, x)
        abi.gate_apply_group([plan, plan, plan], sv, n)
        abi.stream_sync(None)
        got = np.zeros_like(x)
        abi.memcpy_dtoh(got, sv)
    finally:
        abi.free(sv)
        abi.plan_destroy(plan)
    assert np.array_equal(got[rest].view(np.uint64), x[rest].view(np.uint64))
    want = (x[at == row, 0] + 1j * x[at == row, 1]) * -1j
    assert np.allclose(got[at == row, 0] + 1j * got[at == row, 1], want, rtol=1e-15, atol=0)
