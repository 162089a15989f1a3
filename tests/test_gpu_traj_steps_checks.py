"""What a launch per gate step reports about its tables: tasks longer than the
host says, wherever they stand in the order, and (as the persistent launch does)
descriptors that are out of range."""
from __future__ import annotations

import numpy as np
import pytest

from cast_simulator_amd import abi
from test_gpu_traj_steps import Launch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("device,host,flag", [
    ([3, 3], [3, 2], 1), ([3, 2, 1], [3, 2, 0], 1), ([5, 5, 5, 2], [5, 5, 4, 2], 1),
    ([4, 4, 4, 4, 4], [4, 4, 4, 3, 3], 1),  # in the second round of three slots
    ([2] * 3, [0] * 3, 1), ([3, 2, 0], [3, 2, 0], 0), ([3, 2, 1], [4, 4, 2], 0),
])
@pytest.mark.parametrize("n,f64", [(9, True), (12, False)])
def test_longer_tasks_set_the_error_flag(n, f64, device, host, flag):
    """Longer host lengths do no harm: the steps past a task's end leave it."""
    with Launch(n, f64, device, 3, 64, 2, 5) as x:
        print(f"[traj lengths] n={n} device={device} host={host}", flush=True)
        abi.traj_run(x.L)
        want = x.results()
        abi.traj_run_steps(x.L, host)
        got = x.results()
        assert want[0] == 0 and got[0] == flag
        if not flag:
            np.testing.assert_array_equal(got[2], want[2])


@pytest.mark.parametrize("bad", [(0,), (1,), (0, 1), (0, 1, 2)])
@pytest.mark.parametrize("n,f64", [(9, True), (12, False), (14, False)])
def test_invalid_gates_are_left_out(n, f64, bad):
    """Gates out of range (of the first task in the order) are skipped and
    flagged, as in the persistent launch: the others act on the checkpoint."""
    with Launch(n, f64, [3, 3, 2], 3, 64, 2, 11) as x:
        gates = np.zeros(12 * x.L.n_gates, np.uint8)
        abi.memcpy_dtoh(gates, x.L.gates)
        table = (abi.TrajGate * x.L.n_gates).from_buffer(gates)
        for g in bad:
            table[g].matrix_offset = x.L.n_matrix_elems
        abi.memcpy_htod(x.L.gates, gates)
        print(f"[traj invalid] n={n} gates {bad}", flush=True)
        abi.traj_run(x.L)
        want = x.results()
        abi.memcpy_htod(x.L.slots, np.full((3, 2 << n), 7.0, x.dt))  # of other states
        abi.traj_run_steps(x.L, [3, 3, 2])
        got = x.results()
        assert want[0] == 1 and got[0] == 1
        # sums of at most 2^15 terms of about 2^-15 each, in another order
        np.testing.assert_allclose(got[1], want[1], rtol=0, atol=1e-13)
        np.testing.assert_array_equal(got[2], want[2])


@pytest.mark.parametrize("n,f64", [(9, True), (14, False)])
def test_a_task_out_of_range_leaves_its_results(n, f64):
    with Launch(n, f64, [2, 2, 1], 3, 64, 2, 13) as x:
        tasks, order = np.zeros(16 * 3, np.uint8), np.zeros(3, np.uint32)
        abi.memcpy_dtoh(tasks, x.L.tasks)
        abi.memcpy_dtoh(order, x.L.order)
        (abi.TrajTask * 3).from_buffer(tasks)[order[1]].checkpoint = 9
        abi.memcpy_htod(x.L.tasks, tasks)
        x.out[:], x.dump[:] = -3.0, -5.0
        abi.memcpy_htod(x.L.out, x.out)
        abi.memcpy_htod(x.L.dump, x.dump)
        abi.traj_run_steps(x.L, [2, 2, 1])
        flag, out, dump = x.results()
        assert flag == 1
        assert (out[order[1]] == -3.0).all() and (dump[order[1]] == -5.0).all()
        for t in (order[0], order[2]):
            assert abs(out[t][0] - 1.0) <= (1e-13 if f64 else 1e-5)
