"""A state read by one thread while another runs steps of the same solve:
the run's result is that of an undisturbed run, bit for bit, and every state
read is the state after a whole number of steps.  The same for a batch, and
for right-hand sides of a solve that is being read."""
import threading

import numpy as np
import pytest

import dgcuda_amd as dg
from helpers import mesh, problem_for

pytestmark = pytest.mark.gpu

STEPS, READS = 150, 12


def read_during(read, run):
    """States read (at most READS) until run() returns."""
    got, over, failed = [], threading.Event(), []

    def loop():
        try:
            while not over.is_set() and len(got) < READS:
                got.append(read())
        except Exception as ex:  # noqa: BLE001
            failed.append(ex)

    t = threading.Thread(target=loop)
    t.start()
    try:
        run()
    finally:
        over.set()
        t.join()
    assert not failed, failed
    return got


# a small solve (read through one pinned block) and one read in parts
@pytest.mark.parametrize("N,p,prec,n", [(4, 1, dg.DG_FP64, 16), (4, 4, dg.DG_FP32, 20), (1, 2, dg.DG_FP32, 30),
                                        (4, 2, dg.DG_FP64, 170)])
@pytest.mark.parametrize("graph", [True, False])
def test_solver(N, p, prec, n, graph):
    print("read while running", N, p, prec, n, graph, flush=True)

    def fresh():
        s = dg.Solver(mesh(n), problem_for(N), p, prec)
        s.set_kernel(1 if p < 3 else 2)
        s.project_ic()
        return s

    s = fresh()
    states = [s.get_state()]
    for _ in range(STEPS):
        s.run_steps(1, 0.2, dg.DG_RK4, graph)
        states.append(s.get_state())
    known = {x.tobytes() for x in states}
    s = fresh()
    got = read_during(s.get_state, lambda: s.run_steps(STEPS, 0.2, dg.DG_RK4, graph))
    assert np.array_equal(s.get_state(), states[-1])
    assert all(g.tobytes() in known for g in got)


def test_integrate_and_rhs():
    s = dg.Solver(mesh(40), problem_for(4), 2, dg.DG_FP64)
    s.project_ic()
    c0 = s.get_state()
    k0 = s.rhs(c0, 0.01)
    got = read_during(s.get_state, lambda: [np.testing.assert_array_equal(s.rhs(c0, 0.01), k0) for _ in range(20)])
    assert all(np.array_equal(g, c0) for g in got)
    t_end = 100.5 * s.cfl_dt(0.2)
    s.integrate(t_end, 0.2)
    want = s.get_state()
    s.project_ic()
    read_during(s.get_state, lambda: s.integrate(t_end, 0.2))
    assert np.array_equal(s.get_state(), want)


@pytest.mark.parametrize("prec", [dg.DG_FP32, dg.DG_FP64])
def test_batch(prec):
    def fresh():
        b = dg.Batch(prec)
        for i in range(8):
            b.add(mesh(8 + 4 * i), problem_for(4 if i % 2 else 1), 1 + i // 2, 1e30)
        b.project_ic()
        return b

    b = fresh()
    b.run_steps(STEPS, 0.2)
    want = [b.get_state(i) for i in range(8)]
    b = fresh()
    read_during(lambda: [b.get_state(i) for i in range(8)], lambda: b.run_steps(STEPS, 0.2))
    for i in range(8):
        assert np.array_equal(b.get_state(i), want[i]), i
