"""Band Cholesky and its sweeps at the sizes where their blocking can go
wrong: bands of under one block, exact and ragged multiples of 64, the widest
band of the one-launch sweeps (storage width 512) and the first wider one
(a launch per block), one and several samples, one factor shared by samples,
and zero-energy modes on a wide band.  Reference: the oracle's skyline
LDL^T direct solve."""
import numpy as np
import pytest

import msolve_amd as msa
from msolve_amd import _lib as L
from msolve_amd.model import box_mesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def moduli(ns, ne, seed):
    return 2.1e5 * np.exp(0.3 * np.random.default_rng(seed).standard_normal((ns, ne)))


def skyline_direct(m, E):
    ke, bad = O.ke_mesh(m.conn, m.xyz, E, 0.3)
    assert bad == 0
    ri, data = O.skyline_assemble(m.conn, m.dof, m.n_free, ke)
    fac, rc = O.skyline_factorize(ri, data, 1e-15)
    assert rc == 0
    return O.skyline_solve(ri, fac, m.f)


# blocks -> (free DOFs, storage width): under a block, one whole block and a
# remainder, several blocks with a 60- and a 1-block window remainder, the
# widest one-launch band, the narrowest per-block one
SHAPES = [(1, 1, 1), (2, 2, 2), (4, 3, 1), (16, 1, 1), (7, 5, 4), (14, 10, 10), (13, 11, 11)]


@pytest.mark.parametrize("shape", SHAPES)
def test_direct_solve_at_block_edges(ctx, shape):
    # unit cells: a beam's condition number grows with its slenderness, so
    # two FP64 solvers of a 16 x 1 x 1 beam may differ by ~1e6 eps
    m = msa.cantilever(*shape, *[float(v) for v in shape])
    ns = 1 if shape[0] > 12 and shape[1] > 1 else 3
    E = moduli(ns, m.n_elem, sum(shape))
    mesh = msa.Mesh(ctx, m.xyz, m.conn, m.dof, m.n_free)
    b = msa.Batch(ctx, [mesh], [ns], L.MSA_FP64, 0)
    b.set_modulus(0, E)
    b.set_rhs(0, m.f)
    b.set_solver(msa.MSA_SOLVER_DIRECT)
    b.assemble(0.3)
    b.solve()
    info = b.direct_info(0)
    print(f"\n[case] direct {shape}: {info}", flush=True)
    st = b.stats(0)
    assert (st["status"] == msa.MSA_OK).all()
    for s in range(ns):
        assert rel(b.solution(0, s), skyline_direct(m, E[s])) < 1e-10
    if shape == (14, 10, 10):
        assert info["width"] == 512
    if shape == (13, 11, 11):
        assert info["width"] > 512
    b.close()
    mesh.close()


@pytest.mark.parametrize("shape", [(3, 2, 2), (14, 10, 10), (13, 11, 11)])
@pytest.mark.parametrize("precision", [L.MSA_FP64, L.MSA_MIXED])
def test_shared_factor_sweeps(ctx, shape, precision):
    print(f"\n[case] shared factor {shape} precision={precision}", flush=True)
    m = msa.cantilever(*shape)
    ns = 3
    E = moduli(ns, m.n_elem, 7)
    mesh = msa.Mesh(ctx, m.xyz, m.conn, m.dof, m.n_free)
    b = msa.Batch(ctx, [mesh], [ns], precision, 0)
    b.set_preconditioner(msa.MSA_PRECOND_FIRST_SAMPLE)
    b.set_modulus(0, E)
    b.set_rhs(0, m.f)
    b.assemble(0.3)
    b.solve(tol=1e-11 if precision == L.MSA_FP64 else 1e-9, max_it=400, graph_iters=8)
    st = b.stats(0)
    assert (st["status"] == msa.MSA_OK).all(), st
    if precision == L.MSA_FP64:  # its own exact factor: one or two products
        assert st["iters"][0] <= 2
    bar = 1e-9 if precision == L.MSA_FP64 else 1e-8
    for s in range(ns):
        assert rel(b.solution(0, s), skyline_direct(m, E[s])) < bar
    b.close()
    mesh.close()


def test_zero_energy_modes_of_a_wide_band(ctx):
    xyz, conn = box_mesh(12, 11, 11, 12.0, 11.0, 11.0)
    dof, nf = msa.enumerate_dofs(np.zeros((xyz.shape[0], 3), bool))
    E = moduli(1, conn.shape[0], 3)
    mesh = msa.Mesh(ctx, xyz, conn, dof, nf)
    b = msa.Batch(ctx, [mesh], [1], L.MSA_FP64, 0)
    b.set_modulus(0, E)
    b.set_rhs(0, np.random.default_rng(4).standard_normal(nf))
    b.assemble(0.3)
    b.set_solver(L.MSA_SOLVER_DIRECT)
    b.set_zem(1e-3, 8)
    b.solve()
    assert b.direct_info(0)["width"] > 512
    cols, Z = b.zem(0, 0)
    print(f"\n[case] wide zero-energy modes: columns {cols.tolist()}", flush=True)
    assert len(cols) == 6
    scale = np.abs(b.spmv(0, 0, np.eye(1, nf, 0).ravel())).max()
    for j in range(6):
        # a null vector: K z vanishes to rounding (81 terms of |K| |z|)
        assert np.abs(b.spmv(0, 0, Z[j])).max() <= 1e-9 * scale * np.abs(Z[j]).max()
    b.close()
    mesh.close()


@pytest.mark.parametrize("shape,ns", [((4, 4, 4), 5), ((12, 3, 3), 2), ((9, 8, 8), 3)])
def test_factor_memory(ctx, shape, ns):
    """A factorization takes the band storage msa_batch_direct_info reports
    (n W doubles a sample) and a few vectors beside it (right-hand side, the
    second buffer of wide bands, the two permutations)."""
    model = msa.cantilever(*shape, load=-100.0)
    mesh = msa.Mesh(ctx, model.xyz, model.conn, model.dof, model.n_free)
    b = msa.Batch(ctx, [mesh], [ns], L.MSA_FP64, 1)
    b.set_modulus(0, np.full((ns, model.conn.shape[0]), 2.1e5))
    b.set_rhs(0, model.f)
    b.assemble(0.3)
    before, info = b.device_bytes, b.direct_info(0)
    b.factorize()
    extra = b.device_bytes - before - ns * info["bytes_per_sample"]
    print(f"\n[case] {shape} width {info['width']}: {extra / ns / info['n']:.1f} bytes a row beside the band")
    assert 0 <= extra <= ns * info["n"] * 24 + 4096
    b.close()
    mesh.close()
