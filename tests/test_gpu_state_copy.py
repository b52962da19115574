"""State in and out of a solve: the host array comes back unchanged (FP32:
rounded once), whatever the kernel's layout, the element order, and the size
against the copy's pinned blocks and parts; a kernel change carries the state
over.  Exact comparisons: nothing but conversions happens to the values."""
import concurrent.futures

import numpy as np
import pytest

import dgcuda_amd as dg
from helpers import mesh, problem_for, shuffled_mesh

pytestmark = pytest.mark.gpu


def rounded(a, prec):
    return a if prec == dg.DG_FP64 else a.astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("prec", [dg.DG_FP32, dg.DG_FP64])
@pytest.mark.parametrize("N,p,kind", [(1, 0, 1), (1, 1, 1), (1, 1, 2), (1, 4, 1), (1, 4, 2), (1, 5, 1), (4, 0, 1),
                                      (4, 1, 1), (4, 3, 1), (4, 2, 2), (4, 3, 3), (4, 4, 1), (4, 5, 1)])
def test_state_round_trip(N, p, kind, prec):
    for m in (mesh(5), shuffled_mesh(23)):
        s = dg.Solver(m, problem_for(N), p, prec)
        s.set_kernel(kind)
        a = np.random.default_rng(p).standard_normal(s.shape)
        s.set_state(a)
        assert np.array_equal(s.get_state(), rounded(a, prec))
        if p in (1, 2, 3, 4):
            s.set_kernel(2 if kind == 1 else 1)  # another layout, same state
            assert np.array_equal(s.get_state(), rounded(a, prec))


# 48 doubles a square: below and above one block (1 MiB), two blocks, two
# parts (8 MiB), three and four
@pytest.mark.parametrize("nx,ny", [(52, 52), (53, 52), (74, 74), (147, 148), (149, 148), (181, 182), (260, 259)])
def test_state_round_trip_sizes(nx, ny):
    m = dg.Mesh.periodic_jittered(nx, ny, 0.0, 10.0, 0.0, 10.0, 0.1, 1)
    s = dg.Solver(m, problem_for(4), 2, dg.DG_FP32)
    a = np.random.default_rng(nx).standard_normal(s.shape)
    s.set_state(a)
    assert np.array_equal(s.get_state(), rounded(a, dg.DG_FP32))


def test_states_of_several_threads():
    solvers = [dg.Solver(mesh(60 + 30 * i), problem_for(4), 2, dg.DG_FP64) for i in range(4)]
    arrays = [np.random.default_rng(i).standard_normal(s.shape) for i, s in enumerate(solvers)]

    def trip(i):
        for _ in range(5):
            solvers[i].set_state(arrays[i])
            if not np.array_equal(solvers[i].get_state(), arrays[i]):
                return False
        return True

    with concurrent.futures.ThreadPoolExecutor(4) as ex:
        assert all(ex.map(trip, range(4)))
