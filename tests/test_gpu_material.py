"""The material's tables on the device (runs on the GPU): masses and M^-1 of odd and
lopsided boxes against the oracle (sums of at most eight products: 1e-13), and a
second, other material on the same context leaving nothing of the first."""
import numpy as np
import pytest

from hirensi_amd import solver as S
from hirensi_amd.mesh import BoxMesh
from oracle import oracle as O
from tests.helpers import random_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,npml", [((3, 3, 2), (1, 1, 1, 1, 1)), ((9, 4, 7), (1, 4, 1, 2, 3)),
                                        ((6, 11, 5), (2, 1, 3, 1, 1))])
def test_material_tables(shape, npml):
    import torch
    mesh = BoxMesh(*shape, npml=npml, h=(1.0, 1.25, 0.8))
    first, model = random_model(mesh, seed=1), random_model(mesh, seed=2)
    print(f"material {shape} npml={npml}", flush=True)
    ctx = S.Context(mesh, first)
    ctx.set_material(model)
    mr = O.System(mesh, model).diag_m()
    assert np.max(np.abs(ctx.diag_m() - mr) / mr) < 1e-13
    dev = S.Context(mesh, device_ptrs=True)
    t = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    dev.set_material_ptrs(t(model.lam), t(model.mu), t(model.rho))
    x, y = np.random.default_rng(3).standard_normal((2, mesh.neq))
    z = torch.empty(mesh.neq, dtype=torch.float64, device="cuda")
    S.ShellMat(dev, S.HR_K)._apply(0, t(x), t(y), z)
    dev.synchronize()
    assert np.array_equal(z.cpu().numpy(), S.ShellMat(ctx, S.HR_K)._apply(0, x, y, None))
