"""State in and out at the sizes where the copy changes: below and above what
a conversion kernel reaches in one pinned block (1 MiB), and below, at and
above two, three and four parts (8, 12 and 16 MiB), in FP64, whose array goes
in one piece (384 bytes a square); states of several threads in one block
each; a state set and read with nothing in between.  Exact comparisons:
nothing but conversions happens to the values."""
import concurrent.futures

import numpy as np
import pytest

import dgcuda_amd as dg
from helpers import mesh, problem_for, shuffled_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1, 1), (52, 52), (53, 52), (74, 73), (147, 148), (149, 148), (181, 181), (256, 128),
                                   (182, 181), (209, 209), (210, 209)])
def test_round_trip_fp64(nx, ny):
    s = dg.Solver(dg.Mesh.periodic_jittered(nx, ny, 0.0, 10.0, 0.0, 10.0, 0.1, 1), problem_for(4), 2, dg.DG_FP64)
    a = np.random.default_rng(nx).standard_normal(s.shape)
    s.set_state(a)
    assert np.array_equal(s.get_state(), a)


@pytest.mark.parametrize("prec", [dg.DG_FP64, dg.DG_FP32])
@pytest.mark.parametrize("N,p,kind", [(1, 1, 1), (1, 2, 3), (4, 1, 1), (4, 2, 2), (4, 4, 2), (4, 5, 1)])
def test_small_states_of_several_threads(N, p, kind, prec):
    solvers = []
    for i, m in enumerate((mesh(3), mesh(9), shuffled_mesh(12), mesh(17))):
        s = dg.Solver(m, problem_for(N), p, prec)
        s.set_kernel(kind)
        solvers.append(s)
    arrays = [np.random.default_rng(i).standard_normal(s.shape).astype(np.float32).astype(np.float64)
              for i, s in enumerate(solvers)]

    def trip(i):
        for k in range(8):
            solvers[i].set_state(arrays[i] + k)
            want = (arrays[i] + k).astype(np.float32 if prec == dg.DG_FP32 else np.float64).astype(np.float64)
            if not np.array_equal(solvers[i].get_state(), want):
                return False
        return True

    with concurrent.futures.ThreadPoolExecutor(len(solvers)) as ex:
        assert all(ex.map(trip, range(len(solvers))))
