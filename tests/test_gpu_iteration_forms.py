"""Forms of the PCG iteration: a multigrid batch in which one class does not
coarsen leaves the cycle out once only that class's samples are active; every
sample then follows the recurrence it follows in a batch of its own."""
import numpy as np
import pytest

import msolve_amd as msa
from msolve_amd import _lib as L
from msolve_amd.model import box_mesh

pytestmark = pytest.mark.gpu


def solve(ctx, shapes, nsamp, precision, method, tol, **kw):
    meshes, rng = [], np.random.default_rng(2)
    data = {}
    for k, sh in enumerate([(8, 8, 8), (7, 5, 9)]):
        xyz, conn = box_mesh(*sh, *[float(v) for v in sh])
        cons = np.zeros((xyz.shape[0], 3), bool)
        cons[xyz[:, 2] < 1e-12] = True
        dof, nf = msa.enumerate_dofs(cons)
        data[sh] = (xyz, conn, dof, nf, rng.standard_normal(nf),
                    rng.uniform(1.0, 3.0, (nsamp[k], conn.shape[0])))
    for sh in shapes:
        meshes.append(msa.Mesh(ctx, *data[sh][:4]))
    b = msa.Batch(ctx, meshes, [data[sh][5].shape[0] for sh in shapes], precision, 1)
    b.set_preconditioner(L.MSA_PRECOND_MULTIGRID)
    if precision == L.MSA_MIXED:
        b.set_refinement(method)
    for c, sh in enumerate(shapes):
        b.set_modulus(c, data[sh][5])
        b.set_rhs(c, data[sh][4])
    b.assemble(0.3)
    b.solve(tol=tol, max_it=5000, **kw)
    out = {}
    for c, sh in enumerate(shapes):
        st = b.stats(c)
        assert (st["status"] == msa.MSA_OK).all()
        out[sh] = (st["iters"], [b.solution(c, s) for s in range(len(st["iters"]))])
    replays = b.graph_info()["replays"]
    b.close()
    for m in meshes:
        m.close()
    return out, replays


@pytest.mark.parametrize("graph_iters", [0, 2, 12])
@pytest.mark.parametrize("precision,method", [(L.MSA_FP64, 0), (L.MSA_MIXED, L.MSA_REFINE_RELIABLE),
                                              (L.MSA_MIXED, L.MSA_REFINE_RESTART)])
def test_partial_hierarchy_equals_separate_batches(ctx, precision, method, graph_iters):
    cube, odd = (8, 8, 8), (7, 5, 9)
    kw = dict(nsamp=(3, 2), precision=precision, method=method, tol=1e-10, graph_iters=graph_iters)
    both, _ = solve(ctx, [cube, odd], **kw)
    for sh in (cube, odd):
        alone, _ = solve(ctx, [sh], **kw)
        assert np.array_equal(both[sh][0], alone[sh][0])
        for u, v in zip(both[sh][1], alone[sh][1]):
            assert np.array_equal(u, v)
    assert both[odd][0].min() > 2 * both[cube][0].max()  # the cycle was left out for a while


def launches(b, run):
    """Launches of run() by kernel kind (timed, so eager)."""
    b.set_kernel_timing(True)
    run()
    t = b.kernel_timing()
    b.set_kernel_timing(False)
    return {k: v["launches"] for k, v in t.items()}


@pytest.mark.parametrize("dyn", [False, True])
@pytest.mark.parametrize("shape,lengths,roller", [((5, 4, 3), (5.0, 4.0, 3.0), False),
                                                  ((70, 2, 2), (35.0, 1.5, 1.0), True),
                                                  ((1, 9, 8), (1.0, 4.5, 8.0), False)])
def test_mixed_residual_without_hierarchy(ctx, shape, lengths, roller, dyn):
    """Jacobi MIXED batches from 128 chunks on form the FP64 residual
    matrix-free: the first samples against a batch of those alone (too few
    chunks: the coloured residual).  A replacement every 8 iterations is one
    launch there, one per colour here.  Both stop at a true relative residual of
    1e-11; the blocks' condition is below 1e4 (70 x 2 x 2: clamped along the
    side)."""
    xyz, conn = box_mesh(*shape, *lengths)
    cons = np.zeros((xyz.shape[0], 3), bool)
    cons[xyz[:, 1] < 1e-12] = True
    if roller:
        cons[xyz[:, 0] > lengths[0] * (1 - 1e-12), 2] = True
    dof, nf = msa.enumerate_dofs(cons)
    rng = np.random.default_rng(4)
    f, E = rng.standard_normal(nf), rng.uniform(1.0, 3.0, (130, conn.shape[0]))
    out = []
    for ns in (130, 3):
        mesh = msa.Mesh(ctx, xyz, conn, dof, nf)
        b = msa.Batch(ctx, [mesh], [ns], L.MSA_MIXED, 1)
        b.set_modulus(0, E[:ns])
        b.set_rhs(0, f)
        if dyn:
            b.set_dynamics(1e-2, 0.5, 1e-3, 0.25, 0.5, 1e-2)
        b.assemble(0.25)
        b.assemble(0.3)  # the tables follow a new Poisson ratio
        b.solve(tol=1e-11, max_it=5000, graph_iters=8)
        assert (b.stats(0)["status"] == msa.MSA_OK).all()
        u = [b.solution(0, s) for s in range(3)]
        per = 1 if ns == 130 else mesh.info["colours"]
        n = launches(b, lambda: b.solve(tol=1e-11, max_it=5000, graph_iters=8))
        assert n["spmv_dot"] >= 8 and n["residual64"] == per * (n["spmv_dot"] // 8)
        if dyn:
            n = launches(b, lambda: b.newmark(np.ones(1), 0, 1e-8, 5000, 8))
            # the step's right-hand side and first residual too
            assert n["residual64"] == per * (2 + n["spmv_dot"] // 8)
            b.newmark(np.linspace(1.0, 0.5, 4), acc_dir=0, tol=1e-11, max_it=5000, graph_iters=8)
            u += [v for s in range(3) for v in b.dynamic_state(0, s)[:3]]
        out.append(u)
        b.close()
        mesh.close()
    for a, c in zip(*out):
        assert np.linalg.norm(a - c) <= 1e-7 * np.linalg.norm(c)


@pytest.mark.parametrize("precision", [L.MSA_FP64, L.MSA_MIXED])
@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 4, 3), (63, 1, 1), (64, 2, 1), (3, 9, 70)])
def test_small_batch_forms(ctx, shape, precision):
    """One-slice chunks with the split product and folded reductions (a batch
    of one sample) against the form of larger batches, the sample repeated
    beside others past the limit, and the persistent launch.  Same terms in
    the same order but for the partial sums, so the solves agree to their
    stopping residual of 1e-11 times the condition (below 1e5)."""
    xyz, conn = box_mesh(*shape, *[float(v) for v in shape])
    cons = np.zeros((xyz.shape[0], 3), bool)
    cons[xyz[:, 1] < 1e-12] = True
    dof, nf = msa.enumerate_dofs(cons)
    rng = np.random.default_rng(6)
    f, E = rng.standard_normal(nf), rng.uniform(1.0, 3.0, conn.shape[0])
    slices = -(-(nf // 3) // 64)
    out = []
    for ns, persistent in ((1, False), (1, True), (1024 // slices + 1, False)):
        mesh = msa.Mesh(ctx, xyz, conn, dof, nf)
        b = msa.Batch(ctx, [mesh], [ns], precision, 1)
        b.set_matrix_free_product(False)
        b.set_persistent(persistent)
        b.set_modulus(0, np.tile(E, (ns, 1)))
        b.set_rhs(0, f)
        b.assemble(0.3)
        b.solve(tol=1e-11, max_it=5000, graph_iters=8)
        assert (b.stats(0)["status"] == msa.MSA_OK).all()
        out.append((b.solution(0, 0), b.solution(0, ns - 1)))
        b.close()
        mesh.close()
    if precision == L.MSA_FP64:  # the persistent launch serves FP64 and inner solves
        assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(*out[2])
    for o in out[1:]:
        assert np.linalg.norm(o[0] - out[0][0]) <= 1e-6 * np.linalg.norm(out[0][0])


@pytest.mark.parametrize("dyn", [False, True])
@pytest.mark.parametrize("shape,ns,form", [((24, 24, 24), 1, "upper_triangle"),
                                           ((6, 6, 6), 60, "upper_triangle"),
                                           ((5, 6, 6), 128, "matrix_free"),
                                           ((6, 6, 6), 100, "matrix_free")])
def test_persistent_runs_of_one_slice_chunks(ctx, shape, ns, form, dyn):
    """The persistent launch takes four one-slice chunks per workgroup (its
    barriers cost by the workgroup) and gives the bits of the captured
    blocks, with the stored and with the matrix-free product (235, 5, 4 and 5
    slices a sample)."""
    xyz, conn = box_mesh(*shape, *[float(v) for v in shape])
    cons = np.zeros((xyz.shape[0], 3), bool)
    cons[xyz[:, 0] < 1e-12] = True
    dof, nf = msa.enumerate_dofs(cons)
    rng = np.random.default_rng(7)
    f, E = rng.standard_normal(nf), rng.uniform(1.0, 3.0, (ns, conn.shape[0]))
    out = []
    for persistent in (False, True):
        mesh = msa.Mesh(ctx, xyz, conn, dof, nf)
        b = msa.Batch(ctx, [mesh], [ns], L.MSA_FP64, 1)
        b.set_persistent(persistent)
        b.set_modulus(0, E)
        b.set_rhs(0, f)
        if dyn:
            b.set_dynamics(1e-2, 0.5, 1e-3, 0.25, 0.5, 1e-2)
        b.assemble(0.3)
        b.solve(tol=1e-10, max_it=5000, graph_iters=8)
        assert (b.stats(0)["status"] == msa.MSA_OK).all()
        assert b.product_form(0) == form
        out.append((b.stats(0)["iters"], [b.solution(0, s) for s in (0, ns // 2, ns - 1)]))
        if persistent:
            slices = -(-(nf // 3) // 64)
            assert b.persistent_info()["launches"] == 1
            assert b.persistent_info()["workgroups"] <= 8 * -(-(-(-slices // 4) * ns) // 8)
        b.close()
        mesh.close()
    assert np.array_equal(out[0][0], out[1][0])
    for u, v in zip(out[0][1], out[1][1]):
        assert np.array_equal(u, v)
