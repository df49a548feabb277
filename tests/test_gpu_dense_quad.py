"""Matrix-product passes of periodic lines folded twice (even lengths from 112
points): the shortest, lengths with and without a middle row, the edges of the
16-row tiles, the longest; every axis, and the fused x passes."""
import pytest

import test_gpu_dense_transforms as dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [110, 112, 114, 122, 124, 130, 188, 190, 254, 508, 510])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_poisson_solve_per_axis(axis, n):
    dense.test_poisson_solve_per_axis(axis, n, 1)


@pytest.mark.parametrize("Ng,per", [((115, 9, 14), (1, 0, 1)), ((131, 117, 7), (1, 1, 0)), ((9, 7, 189), (0, 1, 1)),
                                    ((181, 99, 131), (1, 0, 0))], ids=lambda v: "x".join(map(str, v)))
def test_fused_x_passes(Ng, per):
    dense.test_fused_x_passes(Ng, per)
