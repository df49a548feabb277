"""Every closed form and its difference between two times, each component, set on
a field of every staggering, against the oracle's point evaluation."""
import pytest

import mif_oracle as mo
from helpers import grids, rel_err

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")

KINDS = ["ZERO", "ES_VELOCITY", "ES_PRESSURE", "ES_GRAD_P", "VT_VELOCITY", "VT_FORCING", "PT_VELOCITY", "PT_PRESSURE",
         "PT_GRAD_P", "LID_1", "LID_2", "CONSTANT"]
# some tens of roundings of terms no larger than the largest value
TOL = 1e-14


@pytest.mark.parametrize("difference", [False, True], ids=["value", "difference"])
@pytest.mark.parametrize("kind", KINDS)
def test_set(kind, difference):
    print(f"[case] function {kind} difference={difference}", flush=True)
    og, gs = grids((9, 13, 11), (1.5, 1.0, 2.0), (-0.5, 0.0, -1.0), 10.0, 1e-3, 1, (0, 1, 0))
    o, ctx = mo.Oracle(og), mif.Context(gs)
    args = {"Re": 10.0, "c": (0.3, -0.2, 0.7)}
    name = "FN_" + kind
    if difference:
        args.update(base=getattr(mo, name), t0=0.2, t1=1.7)
        assert getattr(mo, name) == getattr(mif, name)
        name = "FN_TIME_DIFFERENCE"
    fields = [*ctx.velocity().components, ctx.pressure()]
    for s, field in enumerate(fields):
        for comp in range(3):
            want = o.zeros(s)
            o.set(want, s, mo.make_fn(getattr(mo, name), **args), comp, 0.6, True)
            field.set(mif.function(getattr(mif, name), **args), comp, 0.6)
            assert rel_err(field.download(), want) < TOL
    ctx.close()
