"""Read-back of solved samples: the direct copy (nodes entirely free or fixed,
numbered in node order, one-sample tiles), the extraction kernel of wider
tiles, and the permutation of other numberings and partly held nodes.  Each is
checked through the matrix in the caller's numbering: K u = f, with f random
so that a swapped entry shows.  Then the device scratch the calls share: calls
of growing, shrinking and over-limit size, and two threads at once."""
import threading

import numpy as np
import pytest
import scipy.sparse as sp

import msolve_amd as msa
from msolve_amd import _lib as L
from msolve_amd.model import box_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [L.MSA_FP64, L.MSA_MIXED])
@pytest.mark.parametrize("tile", [1, 4])
@pytest.mark.parametrize("supports", ["node order", "reversed", "roller"])
def test_solution_in_the_callers_numbering(ctx, supports, tile, precision):
    xyz, conn = box_mesh(4, 3, 2, 4.0, 3.0, 2.0)
    cons = np.zeros((xyz.shape[0], 3), bool)
    cons[xyz[:, 0] < 1e-12] = True
    if supports == "roller":
        cons[xyz[:, 0] > 4.0 - 1e-12, 2] = True
    dof, nf = msa.enumerate_dofs(cons)
    if supports == "reversed":
        dof = np.where(dof >= 0, nf - 1 - dof, dof).astype(np.int32)
    ns = 5
    rng = np.random.default_rng(3)
    f = rng.standard_normal(nf)
    E = rng.uniform(1.0, 2.0, (ns, conn.shape[0]))
    mesh = msa.Mesh(ctx, xyz, conn, dof, nf)
    b = msa.Batch(ctx, [mesh], [ns], precision, tile)
    b.set_modulus(0, E)
    b.set_rhs(0, f)
    b.assemble(0.3)
    b.solve(tol=1e-12, max_it=5000)
    for s in range(ns):
        rp, col, val = b.matrix_csr(0, s)
        u = b.solution(0, s)
        r = f - sp.csr_matrix((val, col, rp), (nf, nf)) @ u
        # MIXED reads back an FP32 matrix: 2^-24 per entry, ~100 terms a row
        lim = 1e-10 if precision == L.MSA_FP64 else 1e-4
        assert np.linalg.norm(r) <= lim * np.linalg.norm(f)
        assert np.array_equal(b.modulus(0, s), E[s])
        assert np.array_equal(b.solution(0, s), u)
    b.close()
    mesh.close()


def test_scratch_sizes_and_threads():
    rng = np.random.default_rng(5)
    unit = np.array([[x, y, z] for z in (0, 1) for x, y in ((0, 0), (1, 0), (1, 1), (0, 1))], float)
    big = 26000  # 67.8 MB of scratch, past the 64 MiB a context keeps
    x = unit[None] + rng.uniform(-0.1, 0.1, (big, 8, 3))
    E = rng.uniform(1.0, 2.0, big)
    c = msa.Context(0)
    want, wst = msa.ke_packed(c, x, E, 0.3)
    got = {}

    def work(k, sizes):
        for n in sizes:
            ke, st = msa.ke_packed(c, x[:n], E[:n], 0.3)
            got[k] = got.get(k, True) and np.array_equal(ke, want[:n]) and np.array_equal(st, wst[:n])

    for sizes in ((1, 700, 20, 5000, 3), (2000,) * 20):
        t = [threading.Thread(target=work, args=(k, sizes)) for k in range(2)]
        for v in t:
            v.start()
        for v in t:
            v.join()
        assert got == {0: True, 1: True}
    c.close()
