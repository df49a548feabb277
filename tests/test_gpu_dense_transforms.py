"""Transform passes as matrix products (line lengths without a specialised
kernel, up to 512 wall nodes or 511 periodic points) against the oracle: every
axis and mode at the edges of the 16-row and 8-column tiles, and the x passes
fused with the divergence, the unpack and the FP64 defect.
"""
import numpy as np
import pytest

import mif_oracle as mo
from helpers import PI, grids, rel_err, seeded_normal

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")

# points per line (walls: nodes; periodic: nodes less the duplicated end)
LENGTHS = [(2, 0), (3, 0), (16, 0), (30, 0), (31, 0), (32, 0), (34, 0), (63, 0), (96, 0), (128, 0), (255, 0),
           (287, 0), (512, 0),
           (2, 1), (3, 1), (15, 1), (16, 1), (29, 1), (30, 1), (32, 1), (33, 1), (101, 1), (126, 1), (255, 1),
           (270, 1), (511, 1)]


def tolerance(gs):
    """1e-11 relative, growing with the Laplacian's condition number above
    1e3: the rounding of two FP64 solves differs by that factor."""
    lmax, lmin = 0.0, np.inf
    for a, n in enumerate((gs.Nx_global, gs.Ny_global, gs.Nz_global)):
        per = gs.periodic[a]
        h = (gs.x_size, gs.y_size, gs.z_size)[a] / (n - 1)
        m = n - 1 if per else 2 * (n - 1)
        lam = 2 * (1 - np.cos(2 * np.pi * np.arange(m) / m)) / h ** 2
        lmax += lam.max()
        lmin = min(lmin, lam[1:].min()) if m > 1 else lmin
    return 1e-11 * max(1.0, lmax / lmin / 1e3)


@pytest.mark.parametrize("n,per", LENGTHS, ids=lambda v: str(v))
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_poisson_solve_per_axis(axis, n, per):
    Ng, p3 = [6, 7, 5], [0, 1, 0]
    Ng[axis], p3[axis] = n + per, per
    print(f"[case] dense poisson {Ng} periodic={p3}", flush=True)
    og, gs = grids(Ng, (1.0, 2.0, 1.5), (0.0, -1.0, 0.0), 1.0, 1.0, 1, p3)
    o = mo.Oracle(og)
    b = seeded_normal(tuple(reversed(o.npts)), 20261203)
    ref = b.copy()
    o.poisson_packed(ref)
    ctx = mif.Context(gs)
    p = ctx.pressure()
    own = tuple(slice(p3[a], p3[a] + b.shape[2 - a]) for a in (2, 1, 0))
    host = np.zeros(p.shape)
    host[own] = b
    p.upload(host)
    mif.poisson_solve(p)
    full = np.zeros(p.shape)
    full[own] = ref
    o.apply_periodic(full, 3)
    assert rel_err(p.download(), full) < tolerance(gs)


FUSED = [((32, 18, 20), (0, 0, 0)), ((33, 18, 21), (1, 0, 1)), ((102, 21, 19), (1, 1, 1)), ((287, 9, 14), (0, 1, 0)),
         ((7, 40, 33), (1, 0, 1)),
         # short x lines with a specialised kernel that run as products
         ((33, 20, 18), (0, 0, 0)), ((65, 20, 18), (1, 0, 1)), ((65, 18, 9), (0, 1, 1)), ((97, 12, 14), (1, 0, 1)),
         ((129, 12, 14), (1, 0, 0))]


@pytest.mark.parametrize("Ng,per", FUSED, ids=lambda v: "x".join(map(str, v)))
def test_fused_x_passes(Ng, per):
    """div(u)/dt formed by the x forward pass, phi and its periodic images
    written by the x inverse pass; in the mixed form with one sweep also the
    FP64 defect and the weighted sums, which reach the FP32 storage floor."""
    print(f"[case] dense fused x passes {Ng} periodic={per}", flush=True)
    og, gs = grids(Ng, (2 * PI, 2.0, PI), (0.0, -1.0, 0.0), 1.0, 1.0, 1, per)
    o = mo.Oracle(og)
    dt = 1e-2
    vel32 = [seeded_normal(o.shape(c), 20261220 + c).astype(np.float32).astype(np.float64) for c in range(3)]
    vel = o.velocity()
    for c in range(3):
        vel[c][...] = vel32[c]
    ref = o.zeros(3)
    o.solve_pressure(ref, vel, dt)
    sols = {}
    for name, prec, sweeps, mode in (("fp64", mif.FP64, 0, mif.SOLVE_AUTO), ("s0", mif.MIXED, 0, mif.SOLVE_FP32),
                                     ("s1", mif.MIXED, 1, mif.SOLVE_FP32), ("t64", mif.MIXED, 0, mif.SOLVE_FP64)):
        ctx = mif.Context(gs, precision=prec)
        if prec == mif.MIXED:
            ctx.set_defect_sweeps(sweeps)
            ctx.set_solve_precision(mode)
        v, p = ctx.velocity(), ctx.pressure()
        v.upload(vel32)
        mif.solve_pressure_equation_homogeneous_periodic(p, v, dt)
        sols[name] = p.download()
        ctx.close()
    assert rel_err(sols["fp64"], ref) < tolerance(gs)

    def off(name):
        d, r = sols[name] - sols[name].mean(), ref - ref.mean()
        return float(np.linalg.norm(d - r) / np.linalg.norm(r))

    r32 = ref.astype(np.float32).astype(np.float64)
    floor = float(np.linalg.norm((r32 - r32.mean()) - (ref - ref.mean())) / np.linalg.norm(ref - ref.mean()))
    print("errors", {k: off(k) for k in ("s0", "s1", "t64")}, "floor", floor, flush=True)
    # FP32 transforms amplify their rounding by at most a few units of the
    # condition number's root on these grids; the other two reach FP32 storage
    assert off("s0") < 1e-5
    assert off("s1") < 1.5 * floor
    assert off("t64") < 1.5 * floor
