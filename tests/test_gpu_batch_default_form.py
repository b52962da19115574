"""The launch form a batch takes until one is set: an FP64 batch of one kernel
class its own kernel (more workgroups per CU than the kernel of every class
holds), small batches of several classes one launch; states are those of the
forms that are set, bit for bit."""
import numpy as np
import pytest

import dgcuda_amd as dg
from helpers import mesh, problem_for

pytestmark = pytest.mark.gpu


def run(prec, solves, mode):
    b = dg.Batch(prec)
    if mode is not None:
        b.set_launch_mode(mode)
    for i, (N, p) in enumerate(solves):
        b.add(mesh(6 + 3 * i, seed=i), problem_for(N), p, 1e30)
    b.project_ic()
    b.run_steps(5, 0.2)
    return b.launch_info(), [b.get_state(i) for i in range(len(solves))]


@pytest.mark.parametrize("solves,form", [
    ([(1, 1), (1, 2), (1, 2)], dg.DG_BATCH_PER_CLASS),  # advection lanes
    ([(4, 1), (4, 2)], dg.DG_BATCH_PER_CLASS),          # Euler lanes
    ([(1, 3), (1, 4), (1, 4)], dg.DG_BATCH_PER_CLASS),  # advection tiles
    ([(4, 4), (4, 3)], dg.DG_BATCH_PER_CLASS),          # Euler tiles
    ([(1, 1), (4, 2)], dg.DG_BATCH_ONE_LAUNCH),
    ([(1, 3), (4, 4)], dg.DG_BATCH_ONE_LAUNCH),
    ([(1, 1), (4, 2), (1, 4), (4, 3)], dg.DG_BATCH_ONE_LAUNCH),
])
def test_default_form_fp64(solves, form):
    got, states = run(dg.DG_FP64, solves, None)
    want, ref = run(dg.DG_FP64, solves, form)
    assert got == want
    for a, b in zip(states, ref):
        assert np.array_equal(a, b)


def test_default_form_fp32_one_launch():
    solves = [(1, 3), (1, 4)]
    assert run(dg.DG_FP32, solves, None)[0] == run(dg.DG_FP32, solves, dg.DG_BATCH_ONE_LAUNCH)[0]
