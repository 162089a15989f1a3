"""Pair sums, norms and marginals where their kernels change path: below and
above one chunk of amplitudes, pairs across every part of the amplitude index,
and marginals with few rows per result.

Sums of 2^n non-negative terms that add up to about 1, in f64: both sides
round at most at about (n + 20) eps of that sum, so 1e-13 absolute."""
from __future__ import annotations

import itertools

import numpy as np
import pytest

import cast_simulator_amd as cs
import oracle
from cast_simulator_amd import abi

pytestmark = pytest.mark.gpu


def state(n, f32, seed):
    x = np.asarray(cs.random_statevector(n, seed))
    sv = cs.HipStatevector(n, cs.Precision.F32 if f32 else cs.Precision.F64)
    sv.upload(x)
    return sv, np.asarray(sv.download())


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n", [2, 5, 8, 9, 11, 12, 13, 15])
def test_every_pair_matches_oracle(n, f32):
    sv, x = state(n, f32, 60 + n)
    pairs = list(itertools.combinations(range(n), 2)) + [(n - 1, 0), (1, 1)]
    got = np.asarray(sv.expect_zz([q for p in pairs for q in p]))  # 32 pairs a launch
    want = oracle.expect_zz(x, pairs[:-1])
    assert np.abs(got[:-1] - want).max() <= 1e-13
    norm = float(np.sum(x * x))
    assert abs(got[-1] - norm) <= 1e-13 and abs(sv.norm_squared() - norm) <= 1e-13
    p = abi.F32 if f32 else abi.F64
    some = pairs[:: max(1, len(pairs) // 31)][:31]
    out = abi.malloc(8 * 33)
    scratch = abi.malloc(abi.observe_scratch_bytes(32))
    try:
        abi.observe_async(sv.dptr(), n, p, some, out, scratch)
        host = np.zeros(1 + len(some))
        abi.memcpy_dtoh(host, out)
    finally:
        abi.free(out)
        abi.free(scratch)
    assert abs(host[0] - norm) <= 1e-13
    assert np.abs(host[1:] - oracle.expect_zz(x, some)).max() <= 1e-13


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,measured", [
    (6, [5]), (7, [0, 6]), (11, [10, 0, 3]), (12, [11, 10, 9, 8]), (13, [6, 7, 8]),
    (16, [8, 9, 10, 11, 12, 13, 14, 15]), (16, [0, 1, 2, 3, 4, 5, 6, 7]),
    (16, [15, 3, 9, 0, 12, 6, 7, 1]), (17, list(range(5, 17))), (17, list(range(4, 17))),
    (20, [19, 2, 7]),
])
def test_marginals_match_oracle(n, measured, f32):
    sv, x = state(n, f32, 80 + n)
    got = np.asarray(sv.marginal_probabilities(measured))
    assert np.abs(got - oracle.marginal(x, measured)).max() <= 1e-13


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n", [1, 10, 14, 21, 22])
def test_norm_matches_host_sum(n, f32):
    sv, x = state(n, f32, 90 + n)
    assert abs(sv.norm_squared() - float(np.sum(x * x))) <= 1e-13
