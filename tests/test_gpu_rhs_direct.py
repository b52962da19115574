"""The allocation-free right-hand side's one-launch form, which reads and
writes the caller's arrays itself, against dg_rhs on the same solver (bit for
bit) on every kernel that has it: meshes in the caller's and in the solver's
own order, element counts that divide by no tile, boundary sides.  Arrays
that overlap (in place) take the scratch instead, with the same result."""
import numpy as np
import pytest

import dgcuda_amd as dg
import oracle as orc
from helpers import golden_mesh, mesh, perturbed_state, problem_for, shuffled_mesh
from test_zz_no_alloc import Hip, noalloc_rhs

pytestmark = pytest.mark.gpu

MESHES = {"ordered": lambda: mesh(11), "shuffled": lambda: shuffled_mesh(13), "boundary": lambda: golden_mesh("sv1refined")}
CASES = [(N, p, k) for N in (1, 4) for p in (1, 2, 3, 4) for k in (1, 2, 3)] + [(1, 0, 1), (4, 0, 1), (1, 5, 1)]


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("prec", [dg.DG_FP32, dg.DG_FP64])
def test_direct_rhs_equals_dg_rhs(name, prec):
    hip, m = Hip(), MESHES[name]()
    for N, p, kind in CASES:
        if name == "boundary" and kind == 1 and p > 3:
            continue  # refused
        prob = problem_for(N)
        if name == "boundary":
            prob = dg.supersonic_vortex() if N == 4 else dg.advection_poly(2)
        o = orc.Oracle.from_mesh(m, p, prob)
        u = perturbed_state(o, prob, m.period, seed=p, amp=1e-3)
        s = dg.Solver(m, prob, p, prec)
        s.set_kernel(kind)
        want = s.rhs(u, dt=0.01)
        got = noalloc_rhs(hip, s, u, 0.01)
        print("%s N=%d p=%d kernel %d prec %d: largest difference %.3e"
              % (name, N, p, kind, prec, np.abs(got - want).max()), flush=True)
        assert np.array_equal(got, want), (N, p, kind)


def test_direct_rhs_in_place_and_between_steps():
    hip, m, prob = Hip(), mesh(12), problem_for(4)
    s = dg.Solver(m, prob, 2, dg.DG_FP64)
    s.project_ic()
    s.run_steps(2, 0.3)
    u = s.get_state()
    d = hip.malloc(u.nbytes)
    try:
        hip.put(d, u)
        s.rhs_device_noalloc(d, d, 0.01)
        hip.sync()
        got = hip.get(d, u.shape)
    finally:
        hip.free(d)
    assert np.array_equal(got, s.rhs(u, dt=0.01))
    noalloc_rhs(hip, s, u, 0.01)  # leaves the run's own state and wave speed alone
    f = dg.Solver(m, prob, 2, dg.DG_FP64)
    f.set_kernel(s.kernel())
    f.project_ic()
    f.run_steps(2, 0.3)
    for x in (s, f):
        x.run_steps(2, 0.3)
    a, b = s.get_state(), f.get_state()
    assert np.abs(a - b).max() <= 1e-13 * np.abs(b).max()
