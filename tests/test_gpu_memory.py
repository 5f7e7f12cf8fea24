"""Solves that meet the end of the device memory: a limit on what the context may
still take stands for a full GPU (hr_limit_memory; host-side, no allocation is
tried past it)."""
import numpy as np
import pytest

from hirensi_amd import solver as S
from hirensi_amd.mesh import BoxMesh, receiver_dofs
from oracle import oracle as O
from tests.helpers import random_model, rel_l2

pytestmark = pytest.mark.gpu

NSTEP, DT = 20, 1.0e-4


def _case(nshot, seed=3):
    mesh = BoxMesh(7, 6, 5, npml=(1, 2, 1, 1, 2))
    model = random_model(mesh, seed=seed)
    lo, top = mesh.rd_lo, mesh.NZ - 1
    nodes = [mesh.node_index(2 * lo[0] + 1 + q % 5, 2 * lo[1] + 2, top - q // 5) for q in range(nshot)]
    rec = receiver_dofs(mesh, nodes[:1] + [mesh.node_index(2 * lo[0], 2 * lo[1] + 1, top)])
    src = np.array([mesh.dof(n, q % 3) for q, n in enumerate(nodes)], dtype=np.int64)
    ftab = np.stack([S.time_table(NSTEP, DT, 2, 60.0 + 5 * q) for q in range(nshot)])
    return mesh, model, src, rec, ftab


def _solve(ctx, src, rec, ftab, history=S.HR_HISTORY_STORE, segment=64):
    n = len(src)
    tr = S.explicit_rk4_petsc_pml_3d_shots(ctx, NSTEP, DT, ftab, np.arange(n, dtype=np.int32), src, np.ones(n), rec,
                                           history=history, segment=segment)
    if history == S.HR_HISTORY_NONE:
        return tr
    gl, gm, J = S.explicit_rk4_petsc_pml_3d_adjoint_otd(ctx, NSTEP, DT, rec, 0.5 * tr)
    return tr, gl, gm, J


# doubles that a batch of eight shots may still take: not all state vectors, the state and
# no more, the state and the interface sums but no flux records
@pytest.mark.parametrize("room", ["part of the state", "state", "state and interface sums"])
def test_context_works_after_a_batch_that_does_not_fit(room):
    mesh, model, src, rec, ftab = _case(8)
    ctx, so = S.Context(mesh, model), O.System(mesh, model)
    nn = mesh.nnode
    nf = 9 * nn + nn % 2
    grown = {"part of the state": 7 * 4 * nf, "state": 7 * 9 * nf, "state and interface sums": 7 * (9 * nf + 6 * nn)}[room]
    one = _solve(ctx, src[:1], rec, ftab[:1])
    x, zero = np.random.default_rng(1).standard_normal(mesh.neq), np.zeros(mesh.neq)
    print(f"batch that does not fit: {room}, neq={mesh.neq}", flush=True)
    ctx._check(ctx.L.hr_limit_memory(ctx.h, 8.0 * grown + 65536.0))     # and the small tables of the batch
    with pytest.raises(S.HrError, match="out of memory"):
        _solve(ctx, src, rec, ftab, history=S.HR_HISTORY_NONE)
    for which in (S.HR_K, S.HR_C, S.HR_G):
        for tr in (False, True):
            z = S.ShellMat(ctx, which)._apply(tr, x, zero, None)
            assert rel_l2(z, so.matmult_add(which, x, zero, tr)) < 1e-12, (which, tr)
    ctx._check(ctx.L.hr_limit_memory(ctx.h, -1.0))
    for a, b in zip(_solve(ctx, src[:1], rec, ftab[:1]), one):
        assert np.array_equal(a, b)
    assert np.abs(_solve(ctx, src, rec, ftab)[0]).max() > 0


def _batch(shape, npml, nshot, nstep):
    mesh = BoxMesh(*shape, npml=npml)
    lo, top = mesh.rd_lo, mesh.NZ - 1
    # on the interface and inside, in the PML beside it, and on one node twice
    nodes = [mesh.node_index(2 * lo[0] + q % 4, 2 * lo[1] + 1, top - q // 4 % 3) for q in range(nshot)]
    rec = receiver_dofs(mesh, nodes[:2] + nodes[:1] + [mesh.node_index(1, 2 * lo[1] + 1, top)])
    src = np.array([mesh.dof(n, q % 3) for q, n in enumerate(nodes)], dtype=np.int64)
    ftab = np.stack([S.time_table(nstep, DT, 2, 300.0 + 5 * q) for q in range(nshot)])
    return mesh, random_model(mesh, seed=7), src, rec, ftab


def _gradient(ctx, src, rec, ftab, history, segment):
    n, nstep = len(src), ftab.shape[1]
    tr = S.explicit_rk4_petsc_pml_3d_shots(ctx, nstep, DT, ftab, np.arange(n, dtype=np.int32), src, np.ones(n), rec,
                                           history=history, segment=segment)
    gl, gm, J = S.explicit_rk4_petsc_pml_3d_adjoint_otd(ctx, nstep, DT, rec, 0.5 * tr)
    return tr, gl, gm, J


# a stored and a checkpointed history on one stream, and a batch on two streams
@pytest.mark.parametrize("shape,npml,nshot,nstep,history", [
    ((7, 6, 5), (1, 2, 1, 1, 2), 3, 7, S.HR_HISTORY_STORE), ((6, 7, 5), (1, 4, 2, 2, 1), 1, 8, S.HR_HISTORY_CHECKPOINT),
    ((24, 24, 12), (5,) * 5, 18, 6, S.HR_HISTORY_STORE)])
@pytest.mark.parametrize("graph", [0, 2])
def test_second_record_set_makes_room(shape, npml, nshot, nstep, history, graph):
    """A context that is full but for the second set of flux records gives it back to the
    buffers of a history and an adjoint, and goes on with one set: the same
    arithmetic in a launch per pass, so 1e-13 relative against the two sets.  A set
    holds 12 NN doubles a shot; the limit is less than that short of what the solves
    allocate, so it leaves no other way."""
    mesh, model, src, rec, ftab = _batch(shape, npml, nshot, nstep)
    print(f"one record set {shape} nshot={nshot} history={history} graph={graph}", flush=True)
    two = S.Context(mesh, model)
    two.set_graph(graph)
    ref = _gradient(two, src, rec, ftab, history, 3)
    assert np.abs(ref[1]).max() > 0
    one = S.Context(mesh, model)
    one.set_graph(graph)
    n = len(src)
    run = lambda: S.explicit_rk4_petsc_pml_3d_shots(one, nstep, DT, ftab, np.arange(n, dtype=np.int32), src, np.ones(n),
                                                    rec, history=S.HR_HISTORY_NONE)
    tr = run()
    # of the checkpoints and the adjoint state (54 NN doubles) all but 6 NN fits; of a stored history nothing
    more = one.history_plan(nstep, history, n, 3)[2] + 48.0 * 8 * mesh.nnode * n
    one._check(one.L.hr_limit_memory(one.h, 0.0 if history == S.HR_HISTORY_STORE else more))
    assert np.array_equal(run(), tr)                          # nothing to allocate: both sets
    got = _gradient(one, src, rec, ftab, history, 3)
    for a, b in zip(got, ref):
        assert rel_l2(a, b) < 1e-13
    assert rel_l2(run(), tr) < 1e-13
    x, zero = np.random.default_rng(1).standard_normal(mesh.neq), np.zeros(mesh.neq)
    assert np.array_equal(S.ShellMat(one, S.HR_K)._apply(True, x, zero, None), S.ShellMat(two, S.HR_K)._apply(True, x, zero, None))
