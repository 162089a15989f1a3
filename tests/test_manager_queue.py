"""The kernel manager's queue over a stand-in for the device library
(fake_device.cpp): what is launched, when it is waited for, and on what."""
from __future__ import annotations

import json
import os
import subprocess
import sys
from pathlib import Path

import pytest

TESTS = Path(__file__).resolve().parent

PRELUDE = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
class Counts(ctypes.Structure):
    _fields_ = [(f, ctypes.c_long) for f in
                ("plans", "syncs", "singles", "grouped", "on_freed", "allocs", "fail_alloc",
                 "pays")]
counts = Counts.in_dll(fake, "cast_fake")
import cast_simulator_amd as cs
def graph(n, gates):
    c = cs.QuantumCircuit(n)
    for g in gates:
        c.add(g)
    return cs.CircuitGraph.from_circuit(c)
def snapshot():
    return {f: getattr(counts, f) for f, _ in Counts._fields_}
"""


@pytest.fixture(scope="module")
def fake_lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("fake") / "fake_device.so"
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-fPIC", "-shared",
                    f"-I{TESTS.parent / 'include'}",
                    str(TESTS / "fake_device.cpp"), "-o", str(out)], check=True)
    return out


def run(fake_lib, script):
    """The script's last line of output, as JSON."""
    r = subprocess.run([sys.executable, "-c", PRELUDE + script, str(fake_lib)], cwd=TESTS.parent,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout.splitlines()[-1])


def test_failed_member_copy_leaves_no_gates_queued(fake_lib):
    """An ensemble that fails to copy a member (out of memory) queues nothing
    for the members that go with it: here three that are kept, with gates not
    yet launched, before the copy that fails."""
    out = run(fake_lib, """
n = 10
gates = [cs.QuantumGate.random_unitary([q], q) for q in range(n)]
for q, p in enumerate([0.3, 0.06]):
    gates.append(cs.QuantumGate.depolarizing(q, p))
    gates += [cs.QuantumGate.random_unitary([t], 50 * q + t) for t in range(n)]
sim = cs.Simulator.f64()
counts.fail_alloc = 4
failed = ""
try:
    sim.sample_trajectory(graph(n, gates), cs.TrajectoryOpts([0], 8, 1, 5))
except cs.CastError as e:
    failed = str(e)
sim.simulate(graph(n, gates[:n]))
print(json.dumps([failed, snapshot()]))
""")
    assert "out of memory" in out[0]
    assert out[1]["on_freed"] == 0


def test_untimed_groups_build_no_tuning_candidates(fake_lib):
    """With the autotuner on (the default), gates that run in a pass with others
    take their own plan; candidates are for gates launched by themselves."""
    out = run(fake_lib, """
n = 24
mgr = cs.HipKernelManager(cs.HipKernelGenSpec.f64())
sv = cs.HipStatevector(n, cs.Precision.F64)
ids = [mgr.generate(cs.QuantumGate.random_unitary([q, q + 1], q)) for q in range(8)]
for i in ids:
    mgr.apply(i, sv)
mgr.sync(False)
grouped = snapshot()
tuned = len(mgr.tuning_report())
for i in ids:
    mgr.apply(i, sv)
mgr.sync(True)
print(json.dumps([grouped, tuned, len(mgr.tuning_report()), snapshot()]))
""")
    grouped, tuned, tuned_timed, timed = out
    assert grouped["plans"] == 8 and grouped["grouped"] == 8 and grouped["singles"] == 0
    assert tuned == 0
    assert tuned_timed == 8 and timed["singles"] == 8  # timed work is gate by gate


def test_untimed_single_gates_are_tuned(fake_lib):
    """A gate that no group takes (f64, six qubits) is sampled in untimed work
    until its kernel is chosen."""
    out = run(fake_lib, """
n = 24
mgr = cs.HipKernelManager(cs.HipKernelGenSpec.f64())
sv = cs.HipStatevector(n, cs.Precision.F64)
big = mgr.generate(cs.QuantumGate.random_unitary(list(range(6)), 1))
small = mgr.generate(cs.QuantumGate.random_unitary([0], 2))
chosen = []
for _ in range(12):
    for i in (small, small, big):
        mgr.apply(i, sv)
    mgr.sync(False)
    chosen.append([e["chosen"] for e in mgr.tuning_report()])
print(json.dumps([big, chosen, snapshot()]))
""")
    big, chosen, counts = out
    assert all(len(c) == 1 for c in chosen)
    assert chosen[0] == [-1] and chosen[-1][0] > 0
    assert counts["grouped"] == 24 and counts["singles"] == 12


def test_ensemble_of_large_members_does_not_wait_at_noisy_gates(fake_lib):
    out = run(fake_lib, """
n = 22
gates = [cs.QuantumGate.random_unitary([q], q) for q in range(n)]
for q in range(3):
    gates.append(cs.QuantumGate.depolarizing(q, 0.3))
    gates += [cs.QuantumGate.random_unitary([t], 50 * q + t) for t in range(n)]
sim = cs.Simulator.f64()
sim.sample_trajectory(graph(n, gates), cs.TrajectoryOpts([0], 8, 1, 4))
print(json.dumps(snapshot()))
""")
    assert out["syncs"] == 1 and out["on_freed"] == 0


@pytest.mark.parametrize("pays", [0, 1])
def test_groups_that_do_not_pay_go_gate_by_gate(fake_lib, pays):
    out = run(fake_lib, f"""
counts.pays = {pays}
mgr = cs.HipKernelManager(cs.HipKernelGenSpec.f64())
sv = cs.HipStatevector(24, cs.Precision.F64)
for q in range(3):
    mgr.apply(mgr.generate(cs.QuantumGate.cz(q, q + 9)), sv)
mgr.sync(False)
print(json.dumps(snapshot()))
""")
    assert (out["grouped"], out["singles"]) == ((3, 0) if pays else (0, 3))
