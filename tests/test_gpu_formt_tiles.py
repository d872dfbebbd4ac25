"""FormT at the edges of its kernel's tiles: 60 points along i, 7 rows along j, chunks of k planes, against
the CPU oracle.  Both sides evaluate in the reference's order without FP contraction and differ in the last few
ulps of the cube root (pow() there, cbrt() here) alone, which reach Rhs divided by at most the cancellation of its six fluxes, about 1e3:
bar 1e-12 relative L2."""
import numpy as np
import pytest
import torch

from tosca_amd import case as C
from tests.test_gpu_formt import _case, _compare

pytestmark = pytest.mark.gpu

SIZES = [  # cells along i, j, k
    (2, 2, 2), (59, 5, 3), (60, 6, 2), (61, 7, 3), (62, 6, 2), (63, 7, 3), (64, 8, 4), (120, 3, 3), (121, 15, 2), (126, 3, 3),
    (127, 15, 2), (3, 14, 19),
]


@pytest.mark.parametrize("les,model", [(0, C.LES_DSM), (1, C.LES_SMAGORINSKY), (1, C.LES_DSM)])
@pytest.mark.parametrize("periodic", [(0, 0, 0), (1, 2, 1), (2, 1, 2)])
@pytest.mark.parametrize("n", SIZES)
def test_formt_tile_edges(n, periodic, les, model):
    from tosca_amd import rhs
    lay, mesh, params, f, tp = _case((n[2], n[0], n[1]), periodic, 41, les, model, walls=True)
    assert (lay.mx, lay.my, lay.mz) == tuple(c + 2 for c in n)
    assert _compare(rhs, lay, mesh, params, f, tp, 1.0, 0, f"{n}") <= 1e-12
