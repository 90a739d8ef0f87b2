"""The FP64 matrix-free PCG product (box grids of equal cells, one-sample
tiles): against the stored upper-triangle product and the full image on the
same batch over the grids it accepts (rows shorter and longer than a
wavefront, one or two nodes across, partly constrained blocks, unequal cell
lengths), static and dynamic; what it does not accept keeps the stored
product; the persistent launch gives the same bits.

Both products are FP64 sums of the same terms, so each row agrees to a few
rounding errors of |K||p| and two solves to a residual of 1e-12 agree to
about 1e-12 times the condition number of these small blocks (below 1e4)."""
import numpy as np
import pytest

import msolve_amd as msa
from msolve_amd import _lib as L
from msolve_amd.model import box_mesh

pytestmark = pytest.mark.gpu

NS = 130  # samples of one chunk each: past the 128 chunks the product starts at


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def block(shape, lengths=None, roller=False):
    """Block clamped at x = 0 (roller: the x = end face also held in z)."""
    lengths = lengths or [float(v) for v in shape]
    xyz, conn = box_mesh(*shape, *lengths)
    cons = np.zeros((xyz.shape[0], 3), bool)
    cons[xyz[:, 0] < 1e-12] = True
    if roller:
        cons[xyz[:, 0] > lengths[0] * (1 - 1e-12), 2] = True
    dof, nf = msa.enumerate_dofs(cons)
    f = np.random.default_rng(1).standard_normal(nf)
    return xyz, conn, dof, nf, f


def solve(ctx, blk, ns, E, form, persistent=False, dyn=False):
    xyz, conn, dof, nf, f = blk
    mesh = msa.Mesh(ctx, xyz, conn, dof, nf)
    b = msa.Batch(ctx, [mesh], [ns], L.MSA_FP64, 1)
    b.set_matrix_free_product(form == "matrix_free")
    b.set_symmetric_product(form != "stored")
    b.set_persistent(persistent)
    b.set_modulus(0, E)
    b.set_rhs(0, f)
    if dyn:
        b.set_dynamics(1e-2, 0.5, 1e-3, 0.25, 0.5, 1e-2)
    b.assemble(0.3)
    b.solve(tol=1e-12, max_it=20000, graph_iters=8)
    st = b.stats(0)
    assert (st["status"] == msa.MSA_OK).all()
    got = b.product_form(0)
    u = [b.solution(0, s) for s in range(0, ns, max(1, ns // 4))]
    b.close()
    mesh.close()
    return u, st["iters"], got


GRIDS = [dict(shape=(4, 3, 2)), dict(shape=(3, 1, 1)), dict(shape=(2, 2, 1)),
         dict(shape=(1, 4, 3)), dict(shape=(70, 1, 2), lengths=[4.0, 1.0, 1.0]),
         dict(shape=(5, 4, 3), roller=True),
         dict(shape=(6, 4, 5), lengths=[1.0, 0.3, 2.0])]


@pytest.mark.parametrize("dyn", [False, True])
@pytest.mark.parametrize("grid", GRIDS)
def test_matrix_free_fp64_product(ctx, grid, dyn):
    blk = block(**grid)
    ns = NS
    E = 2.1e5 * np.exp(0.3 * np.random.default_rng(2).standard_normal((ns, blk[1].shape[0])))
    out = {f: solve(ctx, blk, ns, E, f, dyn=dyn)
           for f in ("matrix_free", "upper_triangle", "stored")}
    thin = grid["shape"][0] < 3 or grid["shape"][1] < 2
    assert out["matrix_free"][2] == "matrix_free"
    assert out["upper_triangle"][2] == ("stored" if thin else "upper_triangle")
    assert out["stored"][2] == "stored"
    for f in ("upper_triangle", "stored"):
        d = max(rel(a, b) for a, b in zip(out["matrix_free"][0], out[f][0]))
        print(f"\n[case] {grid} dyn={dyn} vs {f}: {d:.2e}", flush=True)
        assert d < 1e-8
        assert np.abs(out["matrix_free"][1] - out[f][1]).max() <= 3


def test_large_grid_and_persistent(ctx):
    blk = block((33, 31, 34))
    E = 2.1e5 * np.exp(0.3 * np.random.default_rng(3).standard_normal((1, blk[1].shape[0])))
    um, im, fm = solve(ctx, blk, 1, E, "matrix_free")
    us, is_, fs = solve(ctx, blk, 1, E, "upper_triangle")
    up, ip, fp = solve(ctx, blk, 1, E, "matrix_free", persistent=True)
    assert (fm, fs, fp) == ("matrix_free", "upper_triangle", "matrix_free")
    assert rel(um[0], us[0]) < 1e-9 and abs(int(im[0]) - int(is_[0])) <= 3
    assert np.array_equal(um[0], up[0]) and np.array_equal(im, ip)


def test_what_keeps_the_stored_product(ctx):
    # a grid off by more than rounding, a small batch, a loaded matrix, lane tiles
    xyz, conn, dof, nf, f = block((4, 3, 2))
    E = np.full((NS, conn.shape[0]), 2.1e5)
    bent = xyz.copy()
    bent[np.isclose(xyz[:, 0], 2.0), 0] += 1e-12
    assert solve(ctx, (bent, conn, dof, nf, f), NS, E, "matrix_free")[2] != "matrix_free"
    assert solve(ctx, (xyz, conn, dof, nf, f), 4, E[:4], "matrix_free")[2] != "matrix_free"
    mesh = msa.Mesh(ctx, xyz, conn, dof, nf)
    b = msa.Batch(ctx, [mesh], [NS], L.MSA_FP64, 1)
    b.set_modulus(0, E)
    b.set_rhs(0, f)
    b.assemble(0.3)
    rp, col, val = b.matrix_csr(0, 0)
    for s in range(NS):
        b.set_matrix_csr(0, s, rp, col, 2.0 * val)
    b.solve(tol=1e-11, max_it=5000, graph_iters=8)
    assert b.product_form(0) == "upper_triangle"
    u2 = b.solution(0, 5)
    b.assemble(0.3)
    b.solve(tol=1e-11, max_it=5000, graph_iters=8)
    assert b.product_form(0) == "matrix_free"
    assert rel(2.0 * u2, b.solution(0, 5)) < 1e-8
    b.close()
    bt = msa.Batch(ctx, [mesh], [NS], L.MSA_FP64, 2)
    bt.set_modulus(0, E)
    bt.set_rhs(0, f)
    bt.assemble(0.3)
    bt.solve(tol=1e-11, max_it=5000, graph_iters=8)
    assert bt.product_form(0) == "stored"
    bt.close()
    mesh.close()


@pytest.mark.parametrize("precision", [L.MSA_FP64, L.MSA_MIXED])
@pytest.mark.parametrize("beta", [0.0, 1e-3])
@pytest.mark.parametrize("grid", [dict(shape=(8, 6, 4)), dict(shape=(68, 4, 4), lengths=[8.0, 2.0, 2.0]),
                                  dict(shape=(8, 4, 6), roller=True)])
def test_newmark_step_forms(ctx, grid, beta, precision):
    """A Newmark run on a grid of equal cells (right-hand side and first
    residual matrix-free, one launch each) against the same grid with one
    plane moved by 1e-12, which keeps the element-by-element kernels (one
    launch per colour; the MIXED replacements, here every second iteration,
    are matrix-free on both): steps solved to 1e-11
    agree to that, amplified over the steps."""
    xyz, conn, dof, nf, f = block(**grid)
    bent = xyz.copy()
    bent[np.isclose(xyz[:, 1], grid.get("lengths", grid["shape"])[1] / 2), 1] += 1e-12
    ns = NS if precision == L.MSA_FP64 else 3
    E = 2.1e5 * np.exp(0.3 * np.random.default_rng(5).standard_normal((ns, conn.shape[0])))
    acc = 1e3 * np.sin(np.arange(1, 6))
    out = []
    for x in (xyz, bent):
        mesh = msa.Mesh(ctx, x, conn, dof, nf)
        b = msa.Batch(ctx, [mesh], [ns], precision, 1)
        if precision == L.MSA_MIXED:
            b.set_preconditioner(msa.MSA_PRECOND_MULTIGRID)
            assert b.mg_info(0)["levels"] >= 1
        b.set_modulus(0, E)
        b.set_rhs(0, f)
        b.set_dynamics(1e-2, 0.5, beta, 0.25, 0.5, 1e-2)
        b.set_probe(0, nf - 2)
        b.assemble(0.3)
        b.newmark(acc, 1, 1e-11, 20000, 8)
        out.append([(b.history(0, s), *b.dynamic_state(0, s)[:3]) for s in (0, ns - 1)])
        per = 1 if x is xyz else mesh.info["colours"]
        b.set_kernel_timing(True)
        b.newmark(acc[:1], 1, 1e-8, 20000, 8)
        n = {k: v["launches"] for k, v in b.kernel_timing().items()}
        b.set_kernel_timing(False)
        if precision == L.MSA_FP64:
            assert n["residual64"] == per
        else:
            assert n["residual64"] == 2 * per + n["spmv_dot"] // 2
        b.close()
        mesh.close()
    for a, c in zip(*out):
        d = [rel(x, y) for x, y in zip(a, c)]
        print(f"\n[case] newmark {grid} beta={beta} precision={precision}: {d}", flush=True)
        assert d[0] < 1e-8 and d[1] < 1e-8 and d[2] < 1e-6 and d[3] < 1e-6


@pytest.mark.parametrize("dyn", [False, True])
@pytest.mark.parametrize("grid", [dict(shape=(8, 6, 4)), dict(shape=(72, 4, 4), lengths=[8.0, 2.0, 2.0]),
                                  dict(shape=(8, 4, 12), roller=True)])
def test_fp64_cycle_forms(ctx, grid, dyn):
    """One FP64 V-cycle with matrix-free smoothing products against the
    stored values (full image selected): the same sums in another order, a
    few hundred rounding errors through the levels."""
    xyz, conn, dof, nf, f = block(**grid)
    E = 2.1e5 * np.exp(0.3 * np.random.default_rng(6).standard_normal((2, conn.shape[0])))
    mesh = msa.Mesh(ctx, xyz, conn, dof, nf)
    b = msa.Batch(ctx, [mesh], [2], L.MSA_FP64, 1)
    b.set_preconditioner(msa.MSA_PRECOND_MULTIGRID)
    assert b.mg_info(0)["levels"] >= 1
    b.set_modulus(0, E)
    b.set_rhs(0, f)
    if dyn:
        b.set_dynamics(1e-2, 0.5, 1e-3, 0.25, 0.5, 1e-2)
    r = np.random.default_rng(7).standard_normal(nf)
    z = []
    for sym in (True, False, True):
        b.set_symmetric_product(sym)
        b.assemble(0.3)
        b.solve(tol=1e-8, max_it=200, graph_iters=4)
        assert (b.stats(0)["status"] == msa.MSA_OK).all()
        z.append([b.mg_apply(0, s, r) for s in range(2)])
    for s in range(2):
        assert np.array_equal(z[0][s], z[2][s])
        print(f"\n[case] cycle {grid} dyn={dyn}: {rel(z[0][s], z[1][s]):.2e}", flush=True)
        assert rel(z[0][s], z[1][s]) < 1e-11
    b.close()
    mesh.close()


def residual_launches(b, run):
    """FP64 residual and right-hand side launches of run() (eager)."""
    b.set_kernel_timing(True)
    run()
    n = b.kernel_timing()["residual64"]["launches"]
    b.set_kernel_timing(False)
    return n


@pytest.mark.parametrize("offset,free", [(0.0, True), (-0.3, True), (0.5, True), (100.0, False),
                                         (1e4, False), (1e5, False)])
def test_grids_off_the_origin(ctx, offset, free):
    """Far from the origin the rounding of the coordinates makes the cells
    differ, and the forms with one shared element matrix are left out: the
    solution's residual on the assembled matrix stays at the 1e-12 of the
    stopping test plus the recurrence's own drift, a few eps times the
    condition number (below 1e4)."""
    h, n = 0.1, 6
    xyz, conn, dof, nf, f = block((n, n, n), [h * n] * 3)
    mesh = msa.Mesh(ctx, xyz + offset, conn, dof, nf)
    E = 2.1e5 * np.exp(0.3 * np.random.default_rng(2).standard_normal((NS, conn.shape[0])))
    b = msa.Batch(ctx, [mesh], [NS], L.MSA_FP64, 1)
    b.set_modulus(0, E)
    b.set_rhs(0, f)
    b.assemble(0.3)
    b.solve(tol=1e-12, max_it=5000, graph_iters=8)
    assert (b.stats(0)["status"] == msa.MSA_OK).all()
    assert b.product_form(0) == ("matrix_free" if free else "upper_triangle")
    rp, col, val = b.matrix_csr(0, 3)
    u = b.solution(0, 3)
    r = f - np.array([val[rp[i]:rp[i + 1]] @ u[col[rp[i]:rp[i + 1]]] for i in range(nf)])
    print(f"\n[case] offset {offset}: true residual {np.linalg.norm(r) / np.linalg.norm(f):.2e}",
          flush=True)
    assert np.linalg.norm(r) < 5e-12 * np.linalg.norm(f)
    # right-hand side of a Newmark step, and the MIXED residuals: one
    # matrix-free launch each, or one per colour
    b.set_dynamics(1e-2, 0.5, 1e-3, 0.25, 0.5, 1e-2)
    b.assemble(0.3)
    step = lambda: b.newmark(np.array([1.0]), 1, 1e-8, 5000, 0)  # noqa: E731
    assert residual_launches(b, step) == (1 if free else 8)
    b.close()
    b = msa.Batch(ctx, [mesh], [NS], L.MSA_MIXED, 1)
    b.set_modulus(0, E)
    b.set_rhs(0, f)
    b.assemble(0.3)
    k = residual_launches(b, lambda: b.solve(tol=1e-10, max_it=5000, graph_iters=0))
    outer = b.stats(0)["outer"].max()
    assert outer >= 2 and (k < 8 * outer if free else k % 8 == 0)
    b.close()
    mesh.close()


@pytest.mark.parametrize("ns", [830, 1700])
def test_product_over_runs_of_chunks(ctx, ns):
    """Large batches give a workgroup of the FP64 product runs of chunks (5
    chunks a sample: from 4096 of them runs of 2, 2 and 1, from 8192 of 4 and
    1).  The persistent launch takes one chunk at a time: the same bits."""
    blk = block((10, 10, 10))
    E = 2.1e5 * np.exp(0.3 * np.random.default_rng(8).standard_normal((ns, blk[1].shape[0])))
    ua, ia, fa = solve(ctx, blk, ns, E, "matrix_free")
    up, ip, fp = solve(ctx, blk, ns, E, "matrix_free", persistent=True)
    assert (fa, fp) == ("matrix_free", "matrix_free")
    assert np.array_equal(ia, ip)
    for a, c in zip(ua, up):
        assert np.array_equal(a, c)
