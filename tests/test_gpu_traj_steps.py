"""Trajectory tasks with a launch per gate step against the persistent launch
(the same operations on each amplitude) and, where the engine chooses the
steps, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import cast_simulator_amd as cs
from cast_simulator_amd import abi
from test_gpu_trajectory import check_run

pytestmark = pytest.mark.gpu


class Launch:
    """Tasks of random gates on random checkpoints, with their device tables."""

    def __init__(self, n, f64, lengths, n_slots, block, waves, seed):
        rng = np.random.default_rng(seed)
        dt, self.n, self.n_tasks = (np.float64 if f64 else np.float32), n, len(lengths)
        self.dt, self.bufs, pool, n_ckpt = dt, [], [], 2
        kmax = min(n, 4 if f64 else 6 if n >= 12 else 5)
        gates = (abi.TrajGate * max(1, sum(lengths)))()
        for i in range(sum(lengths)):
            k = 1 + int(rng.integers(kmax)) if i else kmax
            K = 1 << k
            u = np.linalg.qr(rng.standard_normal((K, K)) + 1j * rng.standard_normal((K, K)))[0]
            gates[i].matrix_offset, gates[i].k = sum(map(len, pool)) // 2, k
            for b, q in enumerate(sorted(rng.choice(n, k, replace=False).tolist())):
                gates[i].q[b] = q
            pool.append(np.concatenate([u.real.ravel(), u.imag.ravel(), (u.real + u.imag).ravel()])
                        if k >= 4 else u.ravel().view(np.float64))
        tasks, at = (abi.TrajTask * self.n_tasks)(), 0
        order = rng.permutation(self.n_tasks).astype(np.uint32)
        for t, g in zip(order, lengths):
            tasks[t].first_gate, tasks[t].n_gates, tasks[t].checkpoint = at, g, int(rng.integers(n_ckpt))
            at += g
        state = rng.standard_normal((n_ckpt, 2 << n))
        state /= np.sqrt((state**2).sum(1, keepdims=True))
        L = self.L = abi.TrajLaunch()
        L.precision, L.n_qubits, L.n_tasks, L.n_gates = int(f64), n, self.n_tasks, sum(lengths)
        flat = np.concatenate(pool + [np.zeros(2)]).astype(dt)
        L.n_matrix_elems = len(flat) // 2
        L.tasks, L.order = self.dev(np.frombuffer(bytes(tasks), np.uint8)), self.dev(order)
        L.gates, L.matrices = self.dev(np.frombuffer(bytes(gates), np.uint8)), self.dev(flat)
        L.checkpoints, L.n_checkpoints = self.dev(state.astype(dt)), n_ckpt
        L.n_slots, L.block, L.waves_per_simd = n_slots, block, waves
        L.slots = self.dev(np.zeros((n_slots, 2 << n), dt))
        L.n_pairs = 2
        L.pairs[0], L.pairs[1], L.pairs[2], L.pairs[3] = 0, n - 1, 1, 2
        self.out, self.dump = np.zeros((self.n_tasks, 3)), np.zeros((self.n_tasks, 2 << n), dt)
        L.out, L.dump, L.work = self.dev(self.out), self.dev(self.dump), self.dev(np.zeros(2, np.uint32))

    def dev(self, a):
        a = np.ascontiguousarray(a)
        p = abi.malloc(max(a.nbytes, 16))
        self.bufs.append(p)
        abi.memcpy_htod(p, a)
        return p

    def results(self):
        abi.stream_sync(None)
        work, out, dump = np.zeros(2, np.uint32), self.out.copy(), self.dump.copy()
        abi.memcpy_dtoh(work, self.L.work)
        abi.memcpy_dtoh(out, self.L.out)
        abi.memcpy_dtoh(dump, self.L.dump)
        return int(work[1]), out, dump

    def __enter__(self):
        return self

    def __exit__(self, *a):
        for p in self.bufs:
            abi.free(p)


@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("n,lengths,n_slots,block,waves", [
    (3, [2, 1], 2, 64, 2), (9, [4, 3, 3, 1, 0], 2, 64, 2), (10, [5], 3, 512, 2),
    (12, [6, 6, 2], 3, 256, 4), (13, [7, 4, 4, 4, 1], 3, 512, 2), (15, [9, 1], 2, 128, 2),
    (9, [0, 0], 1, 64, 2),
])
def test_steps_equal_the_persistent_launch(f64, n, lengths, n_slots, block, waves):
    with Launch(n, f64, lengths, n_slots, block, waves, 100 * n + len(lengths)) as x:
        print(f"[traj steps] n={n} f64={f64} lengths={lengths} slots={n_slots}", flush=True)
        abi.traj_run(x.L)
        want = x.results()
        abi.traj_run_steps(x.L, lengths)
        got = x.results()
        assert want[0] == 0 and got[0] == 0
        # at most 2^15 terms of about 2^-15 each, added in another order
        np.testing.assert_allclose(got[1], want[1], rtol=0, atol=1e-13)
        np.testing.assert_array_equal(got[2], want[2])


def test_wrong_lengths():
    with Launch(9, True, [3, 2], 2, 64, 2, 1) as x:
        with pytest.raises(abi.AbiError, match="must not increase"):
            abi.traj_run_steps(x.L, [2, 3])
        abi.traj_run_steps(x.L, [1, 1])  # shorter than the tasks
        assert x.results()[0] == 1


@pytest.mark.parametrize("n,prec", [(15, cs.Precision.F64), (16, cs.Precision.F32)])
def test_engine_steps_match_oracle(n, prec):
    """Few tasks on a statevector of 512 KiB: the steps."""
    lc = cs.LayeredCircuit.random_layers(n, 6, 3)
    S = cs.sample_trajectories(lc, cs.NoiseSpec(0.02, 2, 6, 9), 6)
    kmax = 4 if prec == cs.Precision.F64 else 6
    check_run(lc, S, prec, cs.TrajectoryTuning(2, kmax, 512, 1),
              [(i, i + 1) for i in range(n - 1)])
