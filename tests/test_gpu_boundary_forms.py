"""The boundary pass's closed forms (tabulated per axis: Ethier-Steinman and
the velocity-only field; compared per point: the lid; the rest through the
general evaluator) and the tabulated Ethier-Steinman Neumann data, against the
oracle's point evaluation, on every kind of axis."""
import numpy as np
import pytest

import mif_oracle as mo
from helpers import grids, rel_err, seeded_normal

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")

# the tables expand sin(p + q) and exp(2p) into products: a few roundings of
# values of order one, and differences over 2h times h/2 of them
TOL = 1e-14
KINDS = ["ES_VELOCITY", "VT_VELOCITY", "LID_1", "LID_2", "PT_VELOCITY", "CONSTANT"]


@pytest.mark.parametrize("per", [(0, 0, 0), (1, 0, 1), (0, 1, 0), (0, 0, 1)], ids=lambda p: "p" + "".join(map(str, p)))
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("form", ["fp64", "mixed"])
def test_apply_bc(kind, per, form):
    print(f"[case] boundary form {kind} periodic={per} {form}", flush=True)
    og, gs = grids((11, 70, 9), (1.5, 1.0, 2.0), (-0.5, 0.0, -1.0), 1e3, 1e-3, 1, per)
    o = mo.Oracle(og)
    ref = o.velocity()
    for c in range(3):
        ref[c][...] = seeded_normal(o.shape(c), 20261230 + c).astype(np.float32)
    ctx = mif.Context(gs, precision=mif.FP64 if form == "fp64" else mif.MIXED)
    vel = ctx.velocity()
    vel.upload([ref[c] for c in range(3)])
    t = 0.7
    const = (0.3, -0.2, 0.1)
    o.apply_bc(ref, mo.make_fn(getattr(mo, "FN_" + kind), Re=1e3, c=const), t)
    vel.apply_bc(mif.function(getattr(mif, "FN_" + kind), Re=1e3, c=const), t)
    for c, got in enumerate(vel.download()):
        want = ref[c] if form == "fp64" else ref[c].astype(np.float32)
        assert rel_err(got, want) < (TOL if form == "fp64" else 6e-8 + TOL)


@pytest.mark.parametrize("Ng", [(17, 9, 12), (9, 70, 33)], ids=lambda n: "x".join(map(str, n)))
def test_neumann_data_at_a_time(Ng):
    """The stand-alone solve takes the gradient at one time."""
    print(f"[case] tabulated Neumann data {Ng}", flush=True)
    og, gs = grids(Ng, (1.0, 1.0, 2.0), (0.0, 0.0, -1.0), 10.0, 1e-3, 1, (0, 0, 0))
    o = mo.Oracle(og)
    vel, ref = o.velocity(), o.zeros(3)
    for c in range(3):
        vel[c][...] = seeded_normal(o.shape(c), 20261240 + c)
    # the oracle evaluates the Neumann function at t = 0, where the field is
    # exp(+2 d^2 t / Re) times the one at t
    t = 0.4
    fn = mo.make_fn(mo.FN_TIME_DIFFERENCE, Re=10.0, base=mo.FN_ES_GRAD_P, t0=t, t1=3 * t)
    o.solve_pressure(ref, vel, 1e-3, fn)
    ctx = mif.Context(gs)
    v, p = ctx.velocity(), ctx.pressure()
    v.upload([vel[c] for c in range(3)])
    diff = mif.function(mif.FN_TIME_DIFFERENCE, Re=10.0, base=mif.FN_ES_GRAD_P, t0=t, t1=3 * t)
    mif.solve_pressure_equation_non_homogeneous_neumann(p, v, diff, 0.0, 1e-3)
    assert rel_err(p.download(), ref) < 1e-11
    # one time: minus the field at 0.0 by the oracle's own evaluation
    o.solve_pressure(ref, vel, 1e-3, mo.make_fn(mo.FN_ES_GRAD_P, Re=10.0))
    mif.solve_pressure_equation_non_homogeneous_neumann(p, v, mif.function(mif.FN_ES_GRAD_P, Re=10.0), 0.0, 1e-3)
    assert rel_err(p.download(), ref) < 1e-11
