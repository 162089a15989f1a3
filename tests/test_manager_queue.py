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
                ("plans", "syncs", "singles", "grouped", "on_freed", "allocs", "fail_alloc")]
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
