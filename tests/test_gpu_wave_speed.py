"""The maximum cell wave speed a step's last stage leaves for the next step's
dt (partial maxima per workgroup, reduced over their slots): equal to the
wave speed computed afresh from the same state, with fewer and with more
workgroups than slots, and also after a step of the caller's own dt.

Tolerances: the same formula on the same values in FP64 (contraction may
differ by a few roundings); FP32 tiles form it in FP32 with the hardware
reciprocal and square root (about 2 ulp each).
"""
import numpy as np
import pytest

import dgcuda_amd as dg
from helpers import mesh, problem_for

pytestmark = pytest.mark.gpu

TOL = {dg.DG_FP64: 1e-14, dg.DG_FP32: 2e-6}


@pytest.mark.parametrize("N,p,kind,n", [(4, 1, 1, 6), (4, 1, 1, 150), (4, 2, 2, 6), (4, 3, 3, 80), (1, 2, 1, 100)])
@pytest.mark.parametrize("prec", [dg.DG_FP32, dg.DG_FP64])
def test_wave_speed_after_steps(N, p, kind, n, prec):
    m, prob = mesh(n), problem_for(N)
    s = dg.Solver(m, prob, p, prec)
    s.set_kernel(kind)
    s.project_ic()
    s.run_steps(2, 0.3)
    f = dg.Solver(m, prob, p, prec)
    f.set_kernel(kind)
    f.set_state(s.get_state())
    assert abs(s.cfl_dt(0.3) / f.cfl_dt(0.3) - 1) <= TOL[prec]
    # a step with the caller's dt, then steps of the solver's own
    dt = s.cfl_dt(0.3)
    for x in (s, f):
        x.rk_step(dt)
    assert np.array_equal(s.get_state(), f.get_state())
    assert s.cfl_dt(0.3) == f.cfl_dt(0.3)
    s.run_steps(1, 0.3)
    f.set_state(f.get_state())
    f.run_steps(1, 0.3)
    a, b = s.get_state(), f.get_state()
    assert np.isfinite(a).all()
    assert np.abs(a - b).max() <= 10 * TOL[prec] * np.abs(b).max()
