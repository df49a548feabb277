"""Fields reused after a run that blew up: uploads write a field's extents, so
whatever a step left in the padding beyond them stays, and the adjoint's
products read it with a zero factor.  A step and its adjoint from fresh values
must equal those of fresh fields."""
import numpy as np
import pytest

import mif_oracle as mo
from helpers import grids, seeded_normal

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("records", [True, False], ids=["recorded", "fused"])
@pytest.mark.parametrize("per", [(0, 0, 0), (1, 0, 1)], ids=lambda p: "p" + "".join(map(str, p)))
@pytest.mark.parametrize("Ng", [(15, 13, 12), (65, 10, 9)], ids=lambda n: "x".join(map(str, n)))
def test_reused_fields(Ng, per, records, form):
    print(f"[case] padding {form} {Ng} periodic={per} records={records}", flush=True)
    og, gs = grids(Ng, (1.5, 1.0, 2.0), (-0.5, 0.0, -1.0), 1e3, 2e-3, 2, per)
    o = mo.Oracle(og)
    vel0 = [0.1 * seeded_normal(o.shape(c), 20261250 + c) for c in range(3)]
    bar0 = [seeded_normal(o.shape(c), 20261254 + c) for c in range(4)]
    fn = mif.function(mif.FN_ZERO)
    out = []
    for blown in (False, True):
        ctx = mif.Context(gs, precision=mif.FP64 if form == "fp64" else mif.MIXED)
        vel, buf, buf2, un, ubar = (ctx.velocity() for _ in range(5))
        p, pb, pbar = (ctx.pressure() for _ in range(3))
        if blown:
            ctx.set_stage_records(records)
            vel.upload([np.full(o.shape(c), np.nan) for c in range(3)])
            p.upload(np.zeros(o.shape(3)))
            mif.timestep_n(vel, buf, buf2, fn, 0.0, p, pb, 2)
        for field, shape in zip([*vel.components, *buf.components, *buf2.components, p, pb], [0, 1, 2] * 3 + [3, 3]):
            field.upload(np.zeros(o.shape(shape)))
        vel.upload(vel0)
        un.copy_from(vel)
        ctx.set_stage_records(True)
        mif.timestep(vel, buf, buf2, fn, 0.0, p, pb)
        ubar.upload(bar0[:3])
        pbar.upload(bar0[3])
        mif.timestep_adjoint(un, buf, buf2, ubar, pbar, None)
        out.append([*vel.download(), p.download(), *ubar.download(), pbar.download()])
        ctx.close()
    for a, b in zip(*out):
        assert np.isfinite(b).all()
        assert np.array_equal(a, b)
