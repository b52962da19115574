"""Which solves the allocation-free right-hand side refuses does not hang on
the kernel that the automatic choice found faster: up to p = 2 the limit is
that of the lane kernel's layout (FP64 advection p = 1: 1.4 million triangles;
in the tile layout 262,144).  A kernel that the caller set keeps its own
limit."""
import numpy as np
import pytest

import dgcuda_amd as dg
from helpers import mesh, problem_for
from test_zz_no_alloc import Hip, noalloc_rhs

pytestmark = pytest.mark.gpu


def test_automatic_choice_accepts_what_the_lane_kernel_does():
    hip = Hip()
    m = dg.Mesh.periodic_jittered(370, 360, 0.0, 10.0, 0.0, 10.0, 0.1, 1)  # 266,400 triangles
    s = dg.Solver(m, problem_for(1), 1, dg.DG_FP64)
    u = np.random.default_rng(1).standard_normal(s.shape)
    print("kernel", s.kernel(), flush=True)
    assert np.array_equal(noalloc_rhs(hip, s, u, 0.01), s.rhs(u, 0.01))
    s.set_kernel(2)
    with pytest.raises(dg.DGError) as ei:
        noalloc_rhs(hip, s, u, 0.01)
    assert ei.value.code == dg.STATUS_CODES["DG_ERR_BUDGET"]


@pytest.mark.parametrize("prec", [dg.DG_FP32, dg.DG_FP64])
@pytest.mark.parametrize("N,p", [(1, 1), (1, 2), (4, 1), (4, 2)])
def test_overlapping_arrays_of_the_automatic_choice(N, p, prec):
    hip = Hip()
    s = dg.Solver(mesh(14), problem_for(N), p, prec)
    s.project_ic()
    u = s.get_state()
    d = hip.malloc(u.nbytes)
    try:
        hip.put(d, u)
        s.rhs_device_noalloc(d, d, 0.01)
        hip.sync()
        got = hip.get(d, u.shape)
    finally:
        hip.free(d)
    assert np.array_equal(got, s.rhs(u, 0.01))
