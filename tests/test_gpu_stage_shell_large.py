"""Full steps between walls on fields above 32 MB, where the stage kernels store
non-temporally and take the previous projection: with the boundary shell in
their launch (up to 8 M elements) against the boundary pass of its own, and
fused against recorded stages there and above."""
import pytest

import mif_oracle as mo
from helpers import grids, rel_err
from test_gpu_stage_shell import initial, step

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")

SHELL, ABOVE = (167, 162, 171), (207, 203, 205)


def fields(Ng):
    og, gs = grids(Ng, (1.0, 1.0, 2.0), (0.0, 0.0, -1.0), 1e3, 2e-4, 2, (0, 0, 0))
    return (gs, *initial(mo.Oracle(og)))


@pytest.mark.parametrize("records", [False, True], ids=["fused", "recorded"])
def test_shell_against_boundary_pass(records):
    print(f"[case] stage shell {SHELL} records={records}", flush=True)
    gs, vel, p = fields(SHELL)
    a = step(gs, vel, p, "fp64", mif.function(mif.FN_ZERO), records, 2)
    b = step(gs, vel, p, "fp64", mif.function(mif.FN_CONSTANT, c=(0.0, 0.0, 0.0)), records, 2)
    for x, y in zip(a, b):
        assert rel_err(x, y) < 1e-12


@pytest.mark.parametrize("kind", ["ZERO", "ES_VELOCITY", "LID_1"])
@pytest.mark.parametrize("Ng", [SHELL, ABOVE], ids=lambda n: "x".join(map(str, n)))
def test_fused_against_recorded(Ng, kind):
    print(f"[case] stage shell {Ng} {kind}", flush=True)
    gs, vel, p = fields(Ng)
    fn = mif.function(getattr(mif, "FN_" + kind), Re=1e3)
    a, b = (step(gs, vel, p, "fp64", fn, records, 2)[:4] for records in (False, True))
    for x, y in zip(a, b):
        assert rel_err(x, y) < 1e-12
