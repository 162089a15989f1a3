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
