"""The adjoint kernels at the edges of their tiles (30 x 14 outputs per
workgroup and chunks of 2 to 16 planes in k_adj_xb, 64-point items per row in
k_adj_rhs and k_adj_zb), one adjoint step against the oracle's."""
import numpy as np
import pytest

import mif_oracle as mo
from helpers import PI, grids, rel_err

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")

# node counts around multiples of 30 and 14 (points 0..N of an axis), 64 and
# 128 (rows), the smallest grids, and one that takes the longest chunk
CASES = [((3, 3, 3), (0, 0, 0)), ((4, 3, 4), (1, 0, 1)), ((29, 13, 5), (0, 0, 0)), ((30, 14, 7), (0, 0, 0)),
         ((31, 15, 18), (0, 1, 0)), ((60, 28, 6), (1, 0, 1)), ((63, 9, 9), (1, 1, 1)), ((64, 29, 5), (0, 0, 1)),
         ((65, 30, 5), (1, 0, 0)), ((130, 70, 75), (1, 0, 1))]


@pytest.mark.parametrize("Ng,per", CASES, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("form", ["fp64", "mixed"])
def test_adjoint_step(Ng, per, form):
    print(f"[case] adjoint tiles {Ng} periodic={per} {form}", flush=True)
    og, gs = grids(Ng, (2 * PI, 2.0, PI), (0.0, -1.0, 0.0), 50.0, 0.02, 2, per)
    o = mo.Oracle(og)
    rng = np.random.default_rng(11)

    def fields():
        out = o.velocity()
        for c in range(3):
            out[c][...] = rng.standard_normal(out[c].shape).astype(np.float32)
        return out

    un, y2, y3, ubar = fields(), fields(), fields(), fields()
    pbar = rng.standard_normal(o.shape(3)).astype(np.float32).astype(np.float64)
    ctx = mif.Context(gs, precision=mif.FP64 if form == "fp64" else mif.MIXED)
    dev = [ctx.velocity() for _ in range(4)]
    for d, h in zip(dev, (un, y2, y3, ubar)):
        d.upload([h[c] for c in range(3)])
    dp = ctx.pressure()
    dp.upload(pbar)
    fref, fgot = np.zeros(3), np.zeros(3)
    o.timestep_adjoint(un, y2, y3, ubar, pbar, fref)
    mif.timestep_adjoint(*dev, dp, fgot)
    # the mixed form stores its fields in FP32 and solves in FP32: relative
    # rounding of order 1e-6 over the three stages' divergence and solve
    tol = 1e-11 if form == "fp64" else 2e-4
    for c, got in enumerate(dev[3].download()):
        assert rel_err(got, ubar[c]) < tol, ("u_bar", c, rel_err(got, ubar[c]))
    assert rel_err(dp.download(), pbar) < tol, ("p_bar", rel_err(dp.download(), pbar))
    scale = max(np.max(np.abs(fref)), np.sqrt(un[0].size) * 0.02 if form == "mixed" else 0.0)
    assert np.max(np.abs(fgot - fref)) <= tol * scale, (fgot, fref)
