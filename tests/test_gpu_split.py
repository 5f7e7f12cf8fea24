"""The split stage path at the sizes where its kernels' tiles, layers and lists end:
regular domains that do not fill the element pass's 4 x 4 tiles, chunks of one
layer, one per column and in between, sources and receivers on regular-domain
nodes inside and on the interface, in the PML, and more receivers on one block of
the pull than it has threads.  Against the CPU oracle's textbook RK4 at the
parity bar of the time loops (1e-10 relative L2 on traces and gradients)."""
import numpy as np
import pytest

from hirensi_amd import solver as S
from hirensi_amd.mesh import BoxMesh, receiver_dofs
from oracle import oracle as O
from tests.helpers import random_model, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,npml,tz", [((7, 11, 6), (1, 1, 1, 2, 1), 1), ((7, 11, 6), (1, 1, 1, 2, 1), 0),
                                           ((8, 6, 7), (2, 1, 1, 1, 2), 2), ((6, 7, 5), (1, 4, 2, 2, 1), 3),
                                           ((11, 6, 9), (1, 2, 1, 1, 1), 8)])
def test_split_path_at_tile_and_chunk_edges(shape, npml, tz):
    mesh = BoxMesh(*shape, npml=npml)
    model, true = random_model(mesh, seed=4), random_model(mesh, seed=5)
    lo, hi, top = mesh.rd_lo, mesh.rd_hi, mesh.NZ - 1
    ci, cj = lo[0] + hi[0], lo[1] + hi[1]                    # a node in the middle of the regular domain
    nodes = [mesh.node_index(i, j, top) for j in range(2 * lo[1], 2 * hi[1] + 1) for i in range(2 * lo[0], 2 * hi[0] + 1)]
    nodes += [mesh.node_index(ci, cj, top - 1), mesh.node_index(1, cj, top - 2)]
    rec_eq = receiver_dofs(mesh, nodes)
    # the interface corner's DOFs many times over: more entries than a pull block's threads
    rec_eq = np.concatenate([rec_eq, np.repeat(rec_eq[:3], 100)])
    src_eq = np.array([mesh.dof(mesh.node_index(ci, cj, top), 2), mesh.dof(mesh.node_index(ci, cj, top), 2),
                       mesh.dof(mesh.node_index(ci, cj, top - 3), 0), mesh.dof(mesh.node_index(2 * lo[0], cj, top), 1),
                       mesh.dof(mesh.node_index(1, 1, top), 2)], dtype=np.int64)
    src_val = np.array([1.0, 0.25, -0.5, 0.75, 0.5])
    nstep, dt, fr = 90, 1.0e-4, 60.0
    print(f"split path {shape} npml={npml} tz={tz} neq={mesh.neq} receivers={len(rec_eq)}", flush=True)
    B = np.zeros(mesh.neq)
    np.add.at(B, src_eq, src_val)
    row = {int(e): r for r, e in enumerate(mesh.store_eq)}
    inside = np.array([int(e) in row for e in rec_eq])
    rows = np.array([row[int(e)] for e in rec_eq[inside]])
    rec_eq = rec_eq[inside]                                  # the oracle's traces are regular-domain DOFs
    dobs = O.System(mesh, true).forward(B, nstep, dt, lcase=2, fr=fr)[:, rows].copy()
    ctx = S.Context(mesh, model, tz=tz)
    assert ctx.version() == 4
    tr = S.explicit_rk4_petsc_pml_3d(ctx, nstep, dt, S.time_table(nstep, dt, 2, fr), src_eq, src_val, rec_eq)
    gl, gm, _ = S.explicit_rk4_petsc_pml_3d_adjoint_otd(ctx, nstep, dt, rec_eq, dobs)
    so = O.System(mesh, model)
    U = so.forward(B, nstep, dt, lcase=2, fr=fr)
    P = so.adjoint(U, nstep, dt, rec_eq, dobs)
    glr, gmr = so.control(U, P, nstep, dt)
    assert np.abs(U[:, rows]).max() > 0 and np.abs(glr).max() > 0
    assert rel_l2(tr, U[:, rows]) < 1e-10
    assert rel_l2(gl, glr) < 1e-10 and rel_l2(gm, gmr) < 1e-10
    # the fused tile classes take the same stages
    c3 = S.Context(mesh, model, version=3)
    tr3 = S.explicit_rk4_petsc_pml_3d(c3, nstep, dt, S.time_table(nstep, dt, 2, fr), src_eq, src_val, rec_eq)
    assert rel_l2(tr3, tr) < 1e-12


def test_two_streams_match_one_launch():
    """Stages 1 and 3 of a batch with more than 3072 nodal blocks run on two streams,
    those of one shot in one launch; the same arithmetic, so 1e-13 relative."""
    mesh = BoxMesh(24, 24, 12, npml=(5,) * 5)
    model = random_model(mesh, seed=6)
    lo, top, nshot, nstep, dt = mesh.rd_lo, mesh.NZ - 1, 18, 12, 1.0e-4
    nodes = [mesh.node_index(2 * lo[0] + q, 2 * lo[1] + 7, top - q % 2) for q in range(nshot)]
    rec_eq = receiver_dofs(mesh, nodes[::3])
    src_eq = np.array([mesh.dof(n, q % 3) for q, n in enumerate(nodes)], dtype=np.int64)
    ftab = np.stack([S.time_table(nstep, dt, 2, 400.0 + q) for q in range(nshot)])
    one = np.ones(nshot)
    print(f"two streams neq={mesh.neq} nshot={nshot}", flush=True)
    ctx = S.Context(mesh, model)
    tr = S.explicit_rk4_petsc_pml_3d_shots(ctx, nstep, dt, ftab, np.arange(nshot, dtype=np.int32), src_eq, one, rec_eq)
    obs = 0.5 * tr
    gl, gm, _ = S.explicit_rk4_petsc_pml_3d_adjoint_otd(ctx, nstep, dt, rec_eq, obs)
    c1, sl, sm = S.Context(mesh, model), np.zeros(mesh.nnode), np.zeros(mesh.nnode)
    for q in range(nshot):
        t1 = S.explicit_rk4_petsc_pml_3d(c1, nstep, dt, ftab[q], src_eq[q:q + 1], one[:1], rec_eq)
        assert rel_l2(tr[q], t1) < 1e-13, q
        a, b, _ = S.explicit_rk4_petsc_pml_3d_adjoint_otd(c1, nstep, dt, rec_eq, obs[q])
        sl += a
        sm += b
    assert np.abs(sl).max() > 0
    assert rel_l2(gl, sl) < 1e-13 and rel_l2(gm, sm) < 1e-13


@pytest.mark.parametrize("shape,npml,tz", [((7, 11, 6), (1, 1, 1, 2, 1), 1), ((8, 6, 7), (2, 1, 1, 1, 2), 0),
                                           ((6, 7, 5), (1, 4, 2, 2, 1), 3), ((11, 6, 9), (1, 2, 1, 1, 1), 8)])
@pytest.mark.parametrize("which", [S.HR_K, S.HR_C, S.HR_G])
def test_products_at_tile_and_chunk_edges(shape, npml, tz, which):
    """Operator products on the split path, each after another operator's, whose result
    the regular-domain nodes must not keep, against the oracle's assembled matrices."""
    mesh = BoxMesh(*shape, npml=npml)
    model = random_model(mesh, seed=9)
    rng = np.random.default_rng(which)
    x, y = rng.standard_normal(mesh.neq), rng.standard_normal(mesh.neq)
    print(f"products {shape} npml={npml} tz={tz} which={which}", flush=True)
    so, ctx = O.System(mesh, model), S.Context(mesh, model, tz=tz)
    assert ctx.version() == 4
    for tr in (False, True):
        S.ShellMat(ctx, S.HR_K)._apply(tr, 3.0 * x, y, None)
        z = S.ShellMat(ctx, which)._apply(tr, x, y, None)
        assert rel_l2(z - y, so.matmult_add(which, x, np.zeros(mesh.neq), tr)) < 1e-12


@pytest.mark.parametrize("nez,tz", [(449, 0), (500, 0), (470, 1)])
def test_tall_boxes(nez, tz):
    """More element layers than 64 chunks of the fused kernel's default length (or of the
    caller's) hold: the RK4 stages and the central-difference step against the oracle.
    Version 3, which runs those chunks for every stage, refuses and changes nothing."""
    mesh = BoxMesh(3, 4, nez, npml=(1,) * 5)
    model = random_model(mesh, seed=nez)
    top, nstep, dt, fr = mesh.NZ - 1, 6, 1.0e-4, 400.0
    src = np.array([mesh.dof(mesh.node_index(3, 4, top), 2), mesh.dof(mesh.node_index(3, 3, top - 440), 0)], dtype=np.int64)
    rec = receiver_dofs(mesh, [mesh.node_index(3, 4, top - q) for q in (0, 1, 439, 440)])
    print(f"tall box nez={nez} tz={tz} neq={mesh.neq}", flush=True)
    B = np.zeros(mesh.neq)
    B[src] = (1.0, 0.5)
    row = {int(e): r for r, e in enumerate(mesh.store_eq)}
    rows = np.array([row[int(e)] for e in rec])
    so, ctx = O.System(mesh, model), S.Context(mesh, model, tz=tz)
    assert ctx.version() == 4
    tab = S.time_table(nstep, dt, 2, fr)
    ref = so.forward(B, nstep, dt, lcase=2, fr=fr)[:, rows]
    assert np.abs(ref).max() > 0
    before = ctx.tiling()
    with pytest.raises(S.HrError, match="z-chunks"):
        ctx._check(ctx.L.hr_set_tiling(ctx.h, 0, 7, 3))
    assert ctx.tiling() == before
    assert rel_l2(S.explicit_rk4_petsc_pml_3d(ctx, nstep, dt, tab, src, B[src], rec), ref) < 1e-10
    cd = so.cd_forward(B, nstep, dt, lcase=2, fr=fr)[:, rows]
    assert rel_l2(S.explicit_central_difference_3(ctx, nstep, dt, src, B[src], rec, 2, fr), cd) < 1e-10


@pytest.mark.parametrize("shape,npml", [((7, 6, 5), (2, 1, 1, 2, 1)), ((6, 7, 5), (1, 4, 2, 2, 1))])
def test_a_non_finite_entry_reaches_no_more_than_on_the_fused_kernel(shape, npml):
    """Zero coefficients multiply nothing: entries of a product that a NaN or an infinity in
    x makes non-finite on the split path are so on the fused kernel too (also around a
    regular domain of one element)."""
    mesh = BoxMesh(*shape, npml=npml)
    model = random_model(mesh, seed=2)
    rng = np.random.default_rng(3)
    x, zero = rng.standard_normal(mesh.neq), np.zeros(mesh.neq)
    print(f"non-finite entries {shape} npml={npml}", flush=True)
    c4, c3 = S.Context(mesh, model), S.Context(mesh, model, version=3)
    dofs = rng.choice(mesh.neq, 40, replace=False)
    for which in (S.HR_K, S.HR_C, S.HR_G):
        for tr in (False, True):
            reached = 0                                # C and G do not reach regular-domain-only nodes
            for q, d in enumerate(dofs):
                xx = x.copy()
                xx[d] = np.inf if q % 4 == 0 else np.nan
                a, b = (~np.isfinite(S.ShellMat(c, which)._apply(tr, xx, zero, None)) for c in (c4, c3))
                assert not (a & ~b).any(), (which, tr, d)
                reached += b.any()
            assert reached > len(dofs) // 2, (which, tr)
