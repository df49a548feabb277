"""Velocity-only stages that stream their operands past the cache, on either
side of the field size from which they do, against the oracle."""
import pytest

import mif_oracle as mo
from helpers import grids, rel_err

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")


# fields just below and above 40 MB, with ragged tiles on every axis
@pytest.mark.parametrize("forcing", ["VT_FORCING", "CONSTANT"])
@pytest.mark.parametrize("form,Ng", [("fp64", (153, 170, 167)), ("fp64", (201, 167, 163)), ("mixed", (191, 213, 203)),
                                     ("mixed", (233, 215, 217))], ids=lambda v: v if isinstance(v, str) else str(v[0]))
def test_timestep_velocity(form, Ng, forcing):
    print(f"[case] velocity-only step {form} {Ng} {forcing}", flush=True)
    Re = 1e4
    og, gs = grids(Ng, (1.0, 1.0, 1.0), (0.0, 0.0, 0.0), Re, 1e-3, 1, (0, 0, 0))
    o = mo.Oracle(og)
    const = (0.3, -0.2, 0.1)
    ev = mo.make_fn(mo.FN_VT_VELOCITY, Re=Re)
    fo = mo.make_fn(getattr(mo, "FN_" + forcing), Re=Re, c=const)
    vel, buf, rhs = o.velocity(), o.velocity(), o.velocity()
    o.set_velocity(vel, ev, 0.0)
    ctx = mif.Context(gs, precision=mif.FP64 if form == "fp64" else mif.MIXED)
    gvel, gbuf, grhs = ctx.velocity(), ctx.velocity(), ctx.velocity()
    gvel.upload(vel)
    gev = mif.function(mif.FN_VT_VELOCITY, Re=Re)
    gfo = mif.function(getattr(mif, "FN_" + forcing), Re=Re, c=const)
    o.timestep_velocity(vel, buf, rhs, ev, fo, 0.0)
    mif.timestep_velocity(gvel, gbuf, grhs, gev, gfo, 0.0)
    for c, got in enumerate(gvel.download()):
        assert rel_err(got, vel[c]) < (1e-12 if form == "fp64" else 1e-6), c
