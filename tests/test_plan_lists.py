"""KADConvPlan's recorded launches on the host: what a plan keeps per input geometry (no GPU: the launches
are stubbed)."""
import kadconv
from kadconv.fused import KADConvPlan


def _plan():
    return KADConvPlan(kadconv.KADConv(24).eval())


def test_plan_saved_without_lists_loads():
    """A pickled plan's state has no lists (they hold addresses); an older one's has not even the field."""
    plan = _plan()
    state = plan.__getstate__()
    assert state.pop('_lists') == {}
    again = KADConvPlan.__new__(KADConvPlan)
    getattr(again, '__setstate__', again.__dict__.update)(state)
    assert again._lists == {} and again.dim == plan.dim
