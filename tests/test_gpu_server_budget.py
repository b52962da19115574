"""A budget between a request's estimate and what its solve holds (FP32
Euler p = 1 with the lane kernel's records): the request is accepted, and such
requests run one after the other to the end."""
import pytest

import dgcuda_amd as dg
from helpers import problem_for

pytestmark = pytest.mark.gpu


def accepted(budget):
    sv = dg.Server(dg.DG_FP32, max_slots=4, hbm_budget=budget, steps_per_round=4)
    try:
        sv.submit(dg.request(20, 1, 1e-3, problem_for(4), arrival_s=1e9))  # never arrives: only asked
        return True
    except dg.DGError as ex:
        assert ex.code == dg.STATUS_CODES["DG_ERR_BUDGET"]
        return False
    finally:
        sv.close()


def test_budget_of_the_estimate_alone():
    lo, hi = 1 << 10, 1 << 24
    assert not accepted(lo) and accepted(hi)
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if accepted(mid) else (mid, hi)
    sv = dg.Server(dg.DG_FP32, max_slots=4, hbm_budget=hi, steps_per_round=4)
    ids = [sv.submit(dg.request(20, 1, 0.02, problem_for(4), mesh_seed=i)) for i in range(3)]
    sv.drain()
    res = {r.id: r for r in sv.poll(8)}
    sv.close()
    assert all(res[i].status == 0 for i in ids)
    spans = sorted((res[i].admit_s, res[i].finish_s) for i in ids)
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))  # one at a time
