"""A batch's launch forms: its default, one launch, and per class, on small
and large batches, over captured graphs of one and of eight steps and over
direct launches.  The kernels do
the same arithmetic per solve in every form, so results are equal bit for
bit."""
import numpy as np
import pytest

import dgcuda_amd as dg
from helpers import golden_mesh

pytestmark = pytest.mark.gpu


def cases(sizes, boundary):
    out = []
    for i, nx in enumerate(sizes):
        m = dg.Mesh.periodic_jittered(nx, nx, 0.0, 10.0, 0.0, 10.0, 0.1, 3 + i)
        prob = (dg.advection_gaussian(a=(0.7, -0.4), center=(4.0, 6.0), k=0.3) if i % 2
                else dg.euler_vortex(((3.0, 5.0, 5.0),)))
        out.append((m, prob, 1 + (i // 2) % 4))
    if boundary:  # runs its own kernels beside the classes
        out.append((golden_mesh("sv1"), dg.supersonic_vortex(), 2))
    return out


@pytest.mark.parametrize("prec", [dg.DG_FP32, dg.DG_FP64])
@pytest.mark.parametrize("sizes,boundary", [
    ((9, 5, 12, 7, 16, 8, 11, 13), True),      # every class, small
    ((90, 70, 60, 64, 110, 33, 80, 47), False),  # large
    ((20, 21), False),                         # two classes
    ((17,), False),                            # one class
])
def test_forms_agree(prec, sizes, boundary):
    print("batch forms", prec, sizes, flush=True)
    cs = cases(sizes, boundary)
    got = {}
    for mode in (None, dg.DG_BATCH_ONE_LAUNCH, dg.DG_BATCH_PER_CLASS):
        for graph in (True, False):
            b = dg.Batch(prec)
            if mode is not None:
                b.set_launch_mode(mode)
            for m, prob, p in cs:
                b.add(m, prob, p, 1e30)
            b.project_ic()
            b.run_steps(3, 0.3, graph)
            b.run_steps(34, 0.3, graph)  # graphs of eight steps and of one
            got[(mode, graph)] = [b.get_state(k) for k in range(len(cs))]
            b.close()
    ref = got[(dg.DG_BATCH_ONE_LAUNCH, False)]
    for k in range(len(cs)):
        assert np.all(np.isfinite(ref[k]))
        for key, states in got.items():
            assert np.array_equal(states[k], ref[k]), (key, k)
