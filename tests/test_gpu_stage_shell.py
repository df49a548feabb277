"""The boundary shell written in the stage kernel's launch (closed-form data)
against the boundary pass of its own, which general data take: homogeneous data
as FN_ZERO and as a constant of zero; and the closed forms against the oracle.
Ragged tiles, every kind of axis, fused and recorded stages, several steps."""
import itertools

import numpy as np
import pytest

import mif_oracle as mo
from helpers import grids, rel_err, seeded_normal

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")

PERIODIC = list(itertools.product((0, 1), repeat=3))
SIZES = [(67, 13, 10), (9, 66, 7), (3, 4, 5)]


def step(gs, vel0, p0, form, fn, records, nsteps):
    ctx = mif.Context(gs, precision=mif.FP64 if form == "fp64" else mif.MIXED)
    ctx.set_stage_records(records)
    vel, buf, buf2 = ctx.velocity(), ctx.velocity(), ctx.velocity()
    p, pb = ctx.pressure(), ctx.pressure()
    vel.upload(vel0)
    p.upload(p0)
    mif.timestep_n(vel, buf, buf2, fn, 0.0, p, pb, nsteps)
    out = list(vel.download()) + [p.download()]
    if records:  # the stages' own outputs, shells included
        out += list(buf.download()) + list(buf2.download())
    ctx.close()
    return out


def initial(o):
    vel = [0.1 * seeded_normal(o.shape(c), 20261240 + c).astype(np.float32).astype(np.float64) for c in range(3)]
    return vel, 0.1 * seeded_normal(o.shape(3), 20261243).astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("per", PERIODIC, ids=lambda p: "p" + "".join(map(str, p)))
@pytest.mark.parametrize("Ng", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("form", ["fp64", "mixed"])
def test_full_step(form, Ng, per):
    print(f"[case] stage shell {form} {Ng} periodic={per}", flush=True)
    og, gs = grids(Ng, (1.5, 1.0, 2.0), (-0.5, 0.0, -1.0), 1e3, 2e-4, 2, per)
    vel, p = initial(mo.Oracle(og))
    for records in (False, True):
        a = step(gs, vel, p, form, mif.function(mif.FN_ZERO), records, 2)
        b = step(gs, vel, p, form, mif.function(mif.FN_CONSTANT, c=(0.0, 0.0, 0.0)), records, 2)
        for x, y in zip(a, b):
            assert rel_err(x, y) < (1e-12 if form == "fp64" else 1e-5)


@pytest.mark.parametrize("kind", ["ES_VELOCITY", "VT_VELOCITY", "LID_1", "LID_2"])
@pytest.mark.parametrize("per", [(0, 0, 0), (1, 0, 0), (0, 1, 1)], ids=lambda p: "p" + "".join(map(str, p)))
def test_closed_forms(kind, per):
    print(f"[case] stage shell {kind} periodic={per}", flush=True)
    og, gs = grids((21, 12, 19), (1.5, 1.0, 2.0), (-0.5, 0.0, -1.0), 1e3, 1e-4, 1, per)
    o = mo.Oracle(og)
    vel0, p0 = initial(o)
    vel, buf, buf2 = o.velocity(), o.velocity(), o.velocity()
    p, pb = o.zeros(3), o.zeros(3)
    for c in range(3):
        vel[c][...] = vel0[c]
    p[...] = p0
    o.timestep(vel, buf, buf2, mo.make_fn(getattr(mo, "FN_" + kind), Re=1e3), 0.0, p, pb)
    got = step(gs, vel0, p0, "fp64", mif.function(getattr(mif, "FN_" + kind), Re=1e3), False, 1)
    for x, y in zip(got, [vel[0], vel[1], vel[2], p]):
        assert rel_err(x, y) < 1e-10


@pytest.mark.parametrize("Ng", SIZES[:2], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("form", ["fp64", "mixed"])
def test_velocity_step(form, Ng):
    print(f"[case] stage shell velocity-only {form} {Ng}", flush=True)
    og, gs = grids(Ng, (1.5, 1.0, 2.0), (-0.5, 0.0, -1.0), 1e3, 1e-4, 1, (0, 0, 0))
    vel0, _ = initial(mo.Oracle(og))
    out = []
    for fn in (mif.function(mif.FN_ZERO), mif.function(mif.FN_CONSTANT, c=(0.0, 0.0, 0.0))):
        ctx = mif.Context(gs, precision=mif.FP64 if form == "fp64" else mif.MIXED)
        vel, buf, rhs = ctx.velocity(), ctx.velocity(), ctx.velocity()
        vel.upload(vel0)
        for s in range(2):
            mif.timestep_velocity(vel, buf, rhs, fn, mif.function(mif.FN_VT_FORCING, Re=1e3), s * ctx.dt)
        out.append(list(vel.download()) + list(buf.download()))
        ctx.close()
    for x, y in zip(*out):
        assert rel_err(x, y) < (1e-12 if form == "fp64" else 1e-5)
