"""Rounding of the Ethier-Steinman boundary data that come from tables of
one-coordinate functions: on the tangential faces, where the boundary value is
the field's own, their error against extended precision is no larger than that
of the formula evaluated point by point (Field.set)."""
import numpy as np
import pytest

import mif_oracle as mo
from helpers import grids

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")

DOMAINS = [((1.0, 1.0, 2.0), (0.0, 0.0, -1.0)), ((1.5, 1.0, 2.0), (-0.5, 0.0, -1.0)),
           ((2.0, 2.0, 2.0), (-1.0, -1.0, -1.0)), ((6.0, 6.0, 6.0), (-3.0, -3.0, -3.0))]


def velocity(c, xyz):
    """Component c at t = 0 in 80-bit arithmetic."""
    a, d = np.longdouble(np.pi / 4), np.longdouble(np.pi / 2)
    x, y, z = (xyz[(c + q) % 3] for q in range(3))
    return -a * (np.exp(a * x) * np.sin(a * y + d * z) + np.exp(a * z) * np.cos(a * x + d * y))


@pytest.mark.parametrize("domain", range(len(DOMAINS)))
@pytest.mark.parametrize("n", [33, 64, 97])
def test_tangential_faces(n, domain):
    print(f"[case] boundary precision {n} domain {domain}", flush=True)
    size, lo = DOMAINS[domain]
    Ng = (n, n + 1, n - 2)
    _, gs = grids(Ng, size, lo, 1e3, 1e-3, 1, (0, 0, 0))
    ctx = mif.Context(gs)
    fn = mif.function(mif.FN_ES_VELOCITY, Re=1e3)
    point, table = ctx.velocity(), ctx.velocity()
    point.set(fn)
    table.apply_bc(fn, 0.0)
    err, total = np.zeros(2), 0.0
    for c in range(3):
        p, t = point.components[c].download(), table.components[c].download()
        ext = p.shape[::-1]
        xyz = []
        for a in range(3):
            x = lo[a] + size[a] / (Ng[a] - 1) * np.arange(ext[a])
            xyz.append((x - size[a] / (Ng[a] - 1) / 2 if a == c else x).astype(np.longdouble))
        exact = velocity(c, (xyz[0][None, None, :], xyz[1][None, :, None], xyz[2][:, None, None]))
        for a in range(3):
            if a == c:
                continue
            for side in (0, ext[a] - 1):
                # the interior of the face: its edges may belong to another
                face = tuple(side if 2 - q == a else slice(1, p.shape[q] - 1) for q in range(3))
                err += [float(np.sum((f[face] - exact[face]) ** 2)) for f in (p, t)]
                total += float(np.sum(exact[face] ** 2))
    ctx.close()
    rms = np.sqrt(err / total)
    print(f"point by point {rms[0]:.3e}, tables {rms[1]:.3e}", flush=True)
    assert rms[1] <= rms[0]
