"""Batched gates whose plans ask for a kernel variant or for f32 products: the
direct kernel, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
from cast_simulator_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [abi.F64, abi.F32])
@pytest.mark.parametrize("k", [4, 5, 6])
def test_requests_of_a_plan_keep_the_direct_kernel(k, precision):
    rng = np.random.default_rng(k)
    K = 1 << k
    m = np.linalg.qr(rng.standard_normal((K, K)) + 1j * rng.standard_normal((K, K)))[0]
    asks = [dict(variant=abi.VARIANT_DENSE), dict(variant=abi.VARIANT_MFMA),
            dict(flags=abi.FLAG_MFMA_F32)]
    if precision == abi.F64:
        asks.pop()  # f32 only
    for n in (k + 1, k + 4, 13):
        q = sorted(rng.choice(n, k, replace=False).tolist())
        x = np.asarray(cs.random_statevector(n, n))
        plans = [abi.plan_create(m, q, precision, **a) for a in asks]
        svs = [abi.sv_alloc(n, precision) for _ in range(1 + len(asks))]
        try:
            print(f"[batch forced] k={k} precision={precision} n={n}", flush=True)
            for sv in svs:
                abi.sv_upload(sv, x, precision)
            abi.gate_apply(plans[0], svs[0], n)
            abi.gate_apply_batch(plans, svs[1:], [n] * len(plans))
            abi.stream_sync(None)
            want = np.asarray(abi.sv_download(svs[0], n, precision))
            for ask, sv in zip(asks, svs[1:]):
                np.testing.assert_array_equal(np.asarray(abi.sv_download(sv, n, precision)), want,
                                              err_msg=f"{ask} n={n}")
        finally:
            for sv in svs:
                abi.sv_free(sv)
            for p in plans:
                abi.plan_destroy(p)
