"""Matrix-product x passes whose workgroups hold more waves than row tiles:
those waves only load and store.  The grids of other tests have few lines and
thus the most waves; here the wave counts between that and one per row tile
(rounded to a power of two)."""
import pytest

import test_gpu_dense_transforms as dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ng,per", [((18, 131, 130), (1, 0, 1)), ((18, 90, 89), (0, 0, 0)), ((101, 100, 97), (0, 0, 1)),
                                    ((153, 121, 115), (1, 1, 0)), ((180, 99, 131), (0, 0, 0))],
                         ids=lambda v: "x".join(map(str, v)))
def test_fused_x_passes(Ng, per):
    dense.test_fused_x_passes(Ng, per)
