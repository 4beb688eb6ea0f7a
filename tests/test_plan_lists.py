"""KADConvPlan's recorded launches on the host: what a plan keeps per input geometry (no GPU: the launches
are stubbed)."""
import sys
import threading

import pytest
import torch

import kadconv
from kadconv import _ext, fused
from kadconv.fused import KADConvPlan


def _plan():
    return KADConvPlan(kadconv.KADConv(24).eval())


def _stubbed(monkeypatch):
    """A plan whose forward does everything but launch, and the geometries it recorded, in order."""
    plan, recorded = _plan(), []

    class CallList:
        sizes, movable = [0, 0, 8], True

        def __init__(self, run, groups):
            recorded.append(groups[0][0].shape)

        def run(self, *bases):
            pass

    monkeypatch.setattr(_ext, 'CallList', CallList)
    monkeypatch.setattr(plan, '_grouped', lambda x: True)
    monkeypatch.setattr(plan, '_stages_grouped', lambda x, xin, out: ([], [], out))
    return plan, recorded


def test_plan_saved_without_lists_loads():
    """A pickled plan's state has no lists (they hold addresses); an older one's has not even the field."""
    plan = _plan()
    state = plan.__getstate__()
    assert state.pop('_lists') == {}
    again = KADConvPlan.__new__(KADConvPlan)
    getattr(again, '__setstate__', again.__dict__.update)(state)
    assert again._lists == {} and again.dim == plan.dim


def test_a_used_list_stays(monkeypatch):
    """A geometry in use is not dropped for new ones that come and go."""
    plan, recorded = _stubbed(monkeypatch)
    hot = torch.zeros(1, 24, 50, 50)
    for _ in range(3):
        plan.forward(hot)
    for k in range(3 * fused.MAX_LISTS):
        plan.forward(torch.zeros(1, 24, 4 + k, 4))
        plan.forward(hot)
    assert recorded.count(hot.shape) == 1
    assert len(plan._lists) == fused.MAX_LISTS


def test_first_call_records(monkeypatch):
    """A geometry is prepared once, on its first call; one whose pointers cannot be told apart, each time."""
    plan, recorded = _stubbed(monkeypatch)
    x = torch.zeros(1, 24, 6, 4)
    for _ in range(3):
        plan.forward(x)
    assert len(recorded) == 1 and len(plan._lists) == 1
    monkeypatch.setattr(_ext.CallList, 'movable', False)
    for _ in range(3):
        plan.forward(x.new_zeros(1, 24, 7, 4))
    assert len(recorded) == 4 and len(plan._lists) == 1


def test_lists_with_threads(monkeypatch):
    """Threads that call one layer with more geometries than it keeps."""
    plan, _ = _stubbed(monkeypatch)
    xs = [torch.zeros(1, 24, 4 + k, 4) for k in range(3 * fused.MAX_LISTS)]
    failed = []

    def work(first):
        try:
            for k in range(1500):
                plan.forward(xs[(first + 7 * k) % len(xs)])
        except BaseException as e:
            failed.append(e)

    every = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work, args=(11 * t,)) for t in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(every)
    assert not failed, failed[0]
    assert len(plan._lists) == fused.MAX_LISTS


@pytest.mark.parametrize('dim,n,h,w,grouped', [
    (256, 4, 75, 75, True), (256, 16, 50, 50, True), (256, 4, 100, 100, True),    # 1.1k; 1.9k in 320 tiles
    (128, 8, 100, 100, False), (192, 8, 80, 80, False), (256, 5, 100, 100, False),
    (256, 8, 100, 100, False), (32, 16, 100, 100, True)])
def test_grouped_rule(dim, n, h, w, grouped):
    """Which layers run as grouped launches: the full-resolution DSC's work and tiles."""
    plan = KADConvPlan(kadconv.KADConv(dim).eval())
    assert plan._grouped(torch.empty(n, dim, h, w, device='meta')) == grouped
