"""Products of gates over a union of qubits: leaving out exact zeros changes no bit."""
import numpy as np
import pytest

import cast_simulator_amd as cs
from cast_simulator_amd import _host


def dot_order_product(a, b):
    """a @ b with every product formed and summed in index order, real parts apart."""
    re = np.zeros(a.shape)
    im = np.zeros(a.shape)
    with np.errstate(invalid="ignore", over="ignore"):
        for k in range(len(a)):
            x, y = a[:, k : k + 1], b[k : k + 1]
            re += x.real * y.real - x.imag * y.imag
            im += x.real * y.imag + x.imag * y.real
    return re, im


def same(got, want):
    for g, w in ((got.real, want[0]), (got.imag, want[1])):
        assert np.array_equal(np.signbit(g) | np.isnan(g), np.signbit(w) | np.isnan(w))
        assert np.array_equal(g, w, equal_nan=True)


SHAPES = [([0], [0, 1, 2, 3, 4]), ([0, 2, 3, 5, 7], [2]), ([1, 4], [0, 2]), ([3, 5], [3, 5]),
          ([0, 1, 2], [1, 2, 6, 9])]


@pytest.mark.parametrize("qa,qb", SHAPES)
@pytest.mark.parametrize("kind", ["dense", "diagonal", "mixed", "inf", "large", "nan"])
def test_gate_product(qa, qb, kind):
    rng = np.random.default_rng(len(qa) * 100 + len(qb))

    def draw(k, sparse):
        m = rng.standard_normal((2**k, 2**k)) + 1j * rng.standard_normal((2**k, 2**k))
        if sparse:
            m = np.diag(np.diag(m))
        if kind == "inf":
            m[0, -1] = complex(np.inf, 0)
        if kind == "nan":
            m[-1, 0] = complex(np.nan, 1)
        if kind == "large":
            m *= 1e200
        return m

    a = draw(len(qa), kind in ("diagonal", "mixed"))
    b = draw(len(qb), kind == "diagonal")
    got = cs.QuantumGate(a, qa).matmul(cs.QuantumGate(b, qb))
    union = sorted(set(qa) | set(qb))
    assert list(got.qubits()) == union
    ea, eb = _host.expand_matrix(a, qa, union), _host.expand_matrix(b, qb, union)
    for r in range(2 ** len(union)):
        # Expansion by definition: equal outside the gate's qubits, its entry inside.
        for m, q, e in ((a, qa, ea), (b, qb, eb)):
            pos = [union.index(x) for x in q]
            pick = lambda i: sum(((i >> p) & 1) << j for j, p in enumerate(pos))
            rest = ~sum(1 << p for p in pos)
            row = [m[pick(r), pick(c)] if ((r ^ c) & rest) == 0 else 0 for c in range(len(e))]
            assert np.array_equal(e[r], np.array(row), equal_nan=True)
    same(np.asarray(got.matrix()), dot_order_product(ea, eb))
