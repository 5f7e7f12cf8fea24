"""The tiled gradient accumulation at the edges of its tiles (runs on the GPU).

Boxes of one element, of one node column and row more than the 32 x 8 tile, of
several tiles, on random u and p, against the oracle's control pass of one
step.  Bar (FP64, products of derivatives summed in another order): 1e-12 relative
L2; nodes outside the box untouched.
"""
import numpy as np
import pytest

from hirensi_amd import solver as S
from hirensi_amd.mesh import BoxMesh
from oracle import oracle as O
from tests.helpers import random_model, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [(1, 1, 1), (3, 4, 2), (16, 4, 3), (17, 3, 9), (33, 9, 1)])
def test_gradient_tiles(box):
    mesh = BoxMesh(box[0] + 2, box[1] + 2, box[2] + 1, npml=(1,) * 5, h=(1.0, 1.25, 0.8))
    model = random_model(mesh, seed=sum(box))
    print(f"gradient case box={box}", flush=True)
    rng = np.random.default_rng(box[0])
    ns = len(mesh.store_eq)
    U, P = rng.standard_normal((3, ns)), rng.standard_normal((3, ns))
    glr, gmr = O.System(mesh, model).control(U, P, 2, 1.0)
    ctx = S.Context(mesh, model)
    u, p = np.zeros(mesh.neq), np.zeros(mesh.neq)
    u[mesh.store_eq], p[mesh.store_eq] = U[1], P[1]
    gl, gm = np.full(mesh.nnode, 0.5), np.full(mesh.nnode, 0.25)
    out = ~mesh.rd_node.reshape(-1).astype(bool)
    ctx.gradient_accumulate(u, p, 1.0, gl, gm)
    assert np.all(gl[out] == 0.5) and np.all(gm[out] == 0.25)
    assert np.abs(glr).max() > 0
    assert rel_l2(-(gl - 0.5), glr) <= 1e-12 and rel_l2(-(gm - 0.25), gmr) <= 1e-12
