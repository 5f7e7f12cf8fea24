"""The tiled regularisation kernel at the edges of its tiles (runs on the GPU).

Boxes of one element, of whole 4 x 4 tiles, of one element more, and with a last
z-chunk of one layer, against the oracle.  Bars as for the other box sizes (FP64,
only the summation order differs): vectors <= 1e-12 relative L2, costs <= 1e-12
relative; nodes outside the box exactly zero, a second call the same bits.
"""
import numpy as np
import pytest

from hirensi_amd import solver as S
from hirensi_amd.mesh import BoxMesh
from oracle import oracle as O
from tests.helpers import random_model, rel_l2

pytestmark = pytest.mark.gpu

WREG = np.array([50.0, 1.0, 45.0])
BOXES = [(1, 1, 1), (4, 4, 2), (5, 4, 3), (9, 5, 5), (3, 13, 9)]


@pytest.mark.parametrize("box", BOXES)
@pytest.mark.parametrize("method,weighted", [("TV", True), ("TN", False)])
def test_tiles(box, method, weighted):
    mesh = BoxMesh(box[0] + 3, box[1] + 3, box[2] + 1, npml=(1, 2, 2, 1, 1), h=(1.0, 1.25, 0.8))
    model = random_model(mesh, seed=sum(box))
    wreg = WREG if weighted else None
    print(f"tiles case box={box} method={method}", flush=True)
    ctx = S.Context(mesh, model)
    rl, rm, cl, cm = S.regularization(ctx, model.lam, model.mu, method, wreg)
    again = S.regularization(ctx, model.lam, model.mu, method, wreg)
    rlr, rmr, clr, cmr = O.System(mesh, model).regularization(method, model.lam, model.mu, wreg)
    out = ~mesh.rd_node.reshape(-1).astype(bool)
    assert np.abs(rlr).max() > 0 and np.abs(rmr).max() > 0
    assert rel_l2(rl, rlr) <= 1e-12 and rel_l2(rm, rmr) <= 1e-12
    assert abs(cl - clr) <= 1e-12 * abs(clr) and abs(cm - cmr) <= 1e-12 * abs(cmr)
    assert np.all(rl[out] == 0.0) and np.all(rm[out] == 0.0)
    assert np.array_equal(again[0], rl) and np.array_equal(again[1], rm) and again[2:] == (cl, cm)
