"""Single gates on both sides of the sizes from 128 MiB to 16 GiB where the
automatic kernel, its accesses or its tile order change: up to 256 MiB against
the oracle, above against the direct kernel on the device.

Relative L2 of a chain of at most 12 gates <= 1e-12 at f64 (a gate of K <= 64
terms rounds below 1e-14) and <= 1e-5 at f32 (a gate rounds at about 2e-7).
The overlap of two states that differ by a relative d is 1 - d^2 / 2 at least:
1e-12 holds for d <= 1e-6, an amplitude group out of place is at 1e-4 or more."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
import oracle
from cast_simulator_amd import abi
from helpers import rel_l2
from test_gpu_dispatch import low_and_high

pytestmark = pytest.mark.gpu

TOL = {abi.F64: 1e-12, abi.F32: 1e-5}


def unitary(k, rng):
    z = rng.standard_normal((1 << k, 1 << k)) + 1j * rng.standard_normal((1 << k, 1 << k))
    return np.linalg.qr(z)[0]


@pytest.mark.parametrize("precision,n", [(abi.F64, 23), (abi.F64, 24), (abi.F32, 24),
                                         (abi.F32, 25)])
def test_gates_around_the_cache_size(precision, n):
    rng = np.random.default_rng(n + 40 * precision)
    gates = [(unitary(k, rng), low_and_high(k, low, n, rng))
             for k, low in ((1, 0), (3, 0), (3, 3), (4, 0), (4, 2), (4, 3), (5, 1), (5, 3), (6, 2))]
    for k in (1, 2, 6):
        gates.append((np.diag(np.exp(2j * np.pi * rng.random(1 << k))), low_and_high(k, 1, n, rng)))
    x = np.asarray(cs.random_statevector(n, n))
    sv = abi.sv_alloc(n, precision)
    try:
        abi.sv_upload(sv, x, precision)
        for m, q in gates:
            print(f"[dispatch large] n={n} precision={precision} q={q}", flush=True)
            plan = abi.plan_create(m, q, precision)
            abi.gate_apply(plan, sv, n)
            abi.stream_sync(None)
            abi.plan_destroy(plan)
        got = abi.sv_download(sv, n, precision)
    finally:
        abi.sv_free(sv)
    if precision == abi.F32:
        x = x.astype(np.float32)
    oracle.apply_gates(x, gates)
    assert rel_l2(x.astype(np.float64), got) <= TOL[precision]


@pytest.mark.parametrize("precision,n", [(abi.F64, 25), (abi.F64, 27), (abi.F64, 28),
                                         (abi.F64, 30), (abi.F32, 26), (abi.F32, 28),
                                         (abi.F32, 29)])
def test_large_states_equal_the_direct_kernel(precision, n):
    rng = np.random.default_rng(n + 40 * precision)
    f32 = precision == abi.F32
    one, two = (cs.HipStatevector(n, cs.Precision.F32 if f32 else cs.Precision.F64)
                for _ in range(2))
    gates = [(unitary(1, rng), [q], 0) for q in range(n)]  # a state without zeros, on both sides
    gates += [(unitary(k, rng), low_and_high(k, low, n, rng), 1)
              for k, low in ((2, 0), (3, 1), (3, 3), (4, 2), (4, 3), (5, 2))]
    gates += [(unitary(4, rng), list(range(n - 7, n - 3)), 1)]  # neighbouring high targets
    gates += [(np.diag(np.exp(2j * np.pi * rng.random(1 << k))), low_and_high(k, 1, n, rng), 1)
              for k in (1, 3, 6)]
    one.zero()
    two.zero()
    for m, q, automatic in gates:
        print(f"[dispatch large] n={n} precision={precision} q={q}", flush=True)
        direct = abi.plan_create(m, q, precision, variant=abi.VARIANT_DENSE)
        auto = abi.plan_create(m, q, precision) if automatic else direct
        abi.gate_apply(auto, one.dptr(), n)
        abi.gate_apply(direct, two.dptr(), n)
        abi.stream_sync(None)
        abi.plan_destroy(direct)
        if automatic:
            abi.plan_destroy(auto)
    assert abs(one.fidelity(two) - 1.0) <= 1e-12
