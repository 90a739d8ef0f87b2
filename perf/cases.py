"""Performance cases of the framework: what its users run, through the public
entry points of `msolve_amd`, on one GPU.

`listed()` names the cases, `draw(rng)` gives further ones of the same ranges,
`prepare`/`run` are one user program each, `exact` is the same result in plain
64-bit torch, `work` the bytes and operations a pass cannot do without.

Every solve is the clamped block of the Monte Carlo workload: x = 0 held, a
total load of -100 in z on the far face, cubic cells, Poisson ratio 0.3, a
lognormal Karhunen-Loeve modulus of mean 2.1e5 per sample.
"""
import functools
import math

import numpy as np
import torch

import msolve_amd as msa

NU = 0.3
MEAN_E = 2.1e5
LOAD = -100.0
KL_TERMS = 40
KL_CORR = 0.25
MAX_IT = 20000
GAUSS = 0.5773502691896  # the 13-digit abscissa of the element's Gauss rule
# samples per class whose exact result is formed (a 64-bit CG each)
EXACT_SAMPLES = 2

PRECISION = {"fp64": msa.MSA_FP64, "mixed": msa.MSA_MIXED}
PRECOND = {"jacobi": msa.MSA_PRECOND_JACOBI, "multigrid": msa.MSA_PRECOND_MULTIGRID,
           "first_sample": msa.MSA_PRECOND_FIRST_SAMPLE}


# ------------------------------------------------------------------- cases

def listed():
    return [
        # element stiffness matrices of a small mesh (a 10^3 block), the call
        # an assembly on the host makes per model
        {"name": "ke_1000", "kind": "ke", "elements": 1000},
        # the smallest solve: one 10^3 block, FP64 Jacobi-PCG with the
        # solver's default eager launches; latency and launches count
        {"name": "pcg_fp64_10", "kind": "solve", "precision": "fp64", "precond": "jacobi",
         "meshes": "10x10x10", "samples": "1", "cov": 0.3, "tol": 1e-10, "graph_iters": 0},
        # the direct solver: assembly, band Cholesky and solve of one block
        {"name": "direct_16", "kind": "direct", "meshes": "16x16x16", "cov": 0.3},
        # the reference's own Monte Carlo scheme: every sample preconditioned
        # by the factor of the first sample's matrix
        {"name": "mc_first_sample_12", "kind": "solve", "precision": "fp64",
         "precond": "first_sample", "meshes": "12x12x12", "samples": "8", "cov": 0.3,
         "tol": 1e-10, "graph_iters": 12},
        # strains, stresses and forces of one solved 32^3 sample
        {"name": "element_results_32", "kind": "results", "meshes": "32x32x32", "cov": 0.2},
        # odd and ragged block sizes in one mixed batch; the class with odd
        # counts does not coarsen and is solved with Jacobi beside the others
        {"name": "mc_mixed_mg_ragged", "kind": "solve", "precision": "mixed",
         "precond": "multigrid", "meshes": "36x20x12,28x28x10,17x9x13,44x12x6",
         "samples": "5,4,3,4", "cov": 0.5, "tol": 1e-9, "graph_iters": 12},
        # mixed precision with the library's default preconditioner
        {"name": "mc_mixed_jacobi_24", "kind": "solve", "precision": "mixed",
         "precond": "jacobi", "meshes": "24x24x24", "samples": "32", "cov": 0.3, "tol": 1e-9,
         "graph_iters": 12},
        # one large FP64 solve (811 200 unknowns)
        {"name": "pcg_fp64_64", "kind": "solve", "precision": "fp64", "precond": "jacobi",
         "meshes": "64x64x64", "samples": "1", "cov": 0.2, "tol": 1e-10, "graph_iters": 12},
        # a batched FP64 Monte Carlo run, one mesh, Jacobi
        {"name": "mc_fp64_jacobi_32", "kind": "solve", "precision": "fp64", "precond": "jacobi",
         "meshes": "32x32x32", "samples": "64", "cov": 0.2, "tol": 1e-10, "graph_iters": 12},
        # a batched FP64 Monte Carlo run with multigrid over uneven meshes
        {"name": "mc_fp64_mg_uneven", "kind": "solve", "precision": "fp64",
         "precond": "multigrid", "meshes": "16x16x16,24x24x24,32x32x32,48x48x48",
         "samples": "32,32,32,32", "cov": 0.3, "tol": 1e-10, "graph_iters": 12},
        # batched implicit Newmark dynamics, 64 samples of a 48x48x24 block
        # under a 20 Hz base acceleration, mixed multigrid PCG per step
        {"name": "newmark_mixed_mg", "kind": "newmark", "precision": "mixed",
         "precond": "multigrid", "meshes": "48x48x24", "samples": "64", "cov": 0.2,
         "tol": 1e-8, "steps": 20, "rayleigh_alpha": 0.0, "rayleigh_beta": 0.0,
         "graph_iters": 12},
        # the headline: a mixed-precision Monte Carlo run of 1024 samples over
        # five uneven meshes
        {"name": "mc_mixed_mg_1024", "kind": "solve", "precision": "mixed",
         "precond": "multigrid",
         "meshes": "16x16x16,24x24x24,32x32x32,40x40x40,48x48x48",
         "samples": "204,206,212,200,202", "cov": 0.3, "tol": 1e-9, "graph_iters": 12},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi, max_nodes, even):
    """Element counts of a block: each direction over lo..hi, odd ones among
    them unless `even` (multigrid classes halve at least once)."""
    while True:
        d = [_log_int(rng, lo, hi) for _ in range(3)]
        if even:
            d = [max(4, 2 * (v // 2)) for v in d]
        if (d[0] + 1) * (d[1] + 1) * (d[2] + 1) <= max_nodes:
            return d


def _text(boxes):
    return ",".join("x".join(str(v) for v in b) for b in boxes)


def draw(rng):
    """One more case, no dearer than the listed ones: at most half the
    largest's work, Jacobi solves at most that of the listed Jacobi batch."""
    top = {c["name"]: work(c)["flops"] for c in listed()}
    while True:
        case = _draw(rng)
        jacobi = case.get("precond") == "jacobi"
        limit = top["mc_fp64_jacobi_32"] if jacobi else 0.5 * max(top.values())
        if work(case)["flops"] <= limit and _coarse_rows(case) <= 4000:
            return case


def _coarse_rows(case):
    """Free DOFs of the largest coarsest level of a multigrid case: its band
    factor is solved in every cycle of a sample.  Counted twice where many
    cycles run: time steps, or beside a class that does not coarsen."""
    if case.get("precond") != "multigrid":
        return 0
    rows, plain = 0, case["kind"] == "newmark"
    for box in _boxes(case):
        d = list(box)
        while all(v % 2 == 0 and v >= 4 for v in d):
            d = [v // 2 for v in d]
        n = 3 * _nodes(d)
        if d == list(box) or n > 12000:
            plain = True
        else:
            rows = max(rows, n)
    return rows * 2 if plain else rows


def _draw(rng):
    kind = rng.choice(["ke", "direct", "results", "first_sample", "jacobi", "jacobi",
                       "multigrid", "multigrid", "multigrid", "newmark"])
    cov = rng.choice([0.1, 0.2, 0.3, 0.5])
    graph = rng.choice([0, 8, 12, 16])
    if kind == "ke":
        return {"kind": "ke", "elements": _log_int(rng, 100, 30000)}
    if kind == "direct":
        return {"kind": "direct", "meshes": _text([_box(rng, 4, 20, 8000, False)]), "cov": cov}
    if kind == "results":
        return {"kind": "results", "meshes": _text([_box(rng, 6, 40, 40000, False)]), "cov": cov}
    if kind == "first_sample":
        return {"kind": "solve", "precision": rng.choice(["fp64", "mixed"]),
                "precond": "first_sample", "meshes": _text([_box(rng, 4, 14, 2400, False)]),
                "samples": str(_log_int(rng, 2, 12)), "cov": cov, "tol": 1e-9,
                "graph_iters": graph}
    if kind == "newmark":
        box = _box(rng, 8, 48, 40000, True)
        return {"kind": "newmark", "precision": rng.choice(["mixed", "mixed", "fp64"]),
                "precond": "multigrid", "meshes": _text([box]),
                "samples": str(_log_int(rng, 1, 24)), "cov": cov, "tol": 1e-8,
                "steps": _log_int(rng, 3, 20),
                "rayleigh_alpha": rng.choice([0.0, 1.0]),
                "rayleigh_beta": rng.choice([0.0, 1e-6]), "graph_iters": graph}
    classes = rng.choice([1, 1, 2, 3])
    if kind == "jacobi":
        boxes = [_box(rng, 8, 64, 120000, False) for _ in range(classes)]
        counts = [_log_int(rng, 1, 32) for _ in range(classes)]
        precision = rng.choice(["fp64", "mixed"])
    else:
        # one block in four has odd counts and stays with Jacobi in the batch
        boxes = [_box(rng, 8, 56, 120000, rng.random() < 0.75) for _ in range(classes)]
        counts = [_log_int(rng, 1, 96) for _ in range(classes)]
        precision = rng.choice(["mixed", "mixed", "fp64"])
    return {"kind": "solve", "precision": precision, "precond": kind, "meshes": _text(boxes),
            "samples": ",".join(str(c) for c in counts), "cov": cov,
            "tol": 1e-10 if precision == "fp64" else 1e-9, "graph_iters": graph}


def _boxes(case):
    return [tuple(int(v) for v in m.split("x")) for m in case["meshes"].split(",")]


def _counts(case):
    return [int(s) for s in case.get("samples", "1").split(",")]


# ----------------------------------------------------------------- inputs

def _lengths(box):
    """Block lengths for cubic cells, 1 in x."""
    return (1.0, box[1] / box[0], box[2] / box[0])


@functools.lru_cache(maxsize=64)
def _kl_1d(length):
    """1-D modes of the exponential covariance on [-L/2, L/2]: frequencies,
    eigenvalues and normalisations, cosine modes at odd 1-based positions."""
    half, c = 0.5 * length, 1.0 / KL_CORR
    k = np.arange(KL_TERMS)
    m = k // 2
    cosine = k % 2 == 0
    lo = np.where(cosine, m * np.pi, (m + 0.5) * np.pi) / half
    hi = np.where(cosine, (m + 0.5) * np.pi, (m + 1.0) * np.pi) / half

    def g(w):
        s, co = np.sin(w * half), np.cos(w * half)
        return np.where(cosine, c * co - w * s, w * co + c * s)

    a, b = lo.copy(), hi.copy()
    sign = np.sign(g(a + 1e-13 / half))
    for _ in range(200):
        w = 0.5 * (a + b)
        left = np.sign(g(w)) == sign
        a, b = np.where(left, w, a), np.where(left, b, w)
    w = 0.5 * (a + b)
    s2 = np.sin(2.0 * w * half) / (2.0 * w)
    norm = 1.0 / np.sqrt(np.where(cosine, half + s2, half - s2))
    return w, 2.0 * c / (w * w + c * c), norm


@functools.lru_cache(maxsize=64)
def _kl_table(lengths):
    """The separable 3-D table of the KL_TERMS largest product eigenvalues."""
    w, lam, a = zip(*(_kl_1d(l) for l in lengths))
    prod = lam[0][:, None, None] * lam[1][None, :, None] * lam[2][None, None, :]
    order = np.argsort(-prod, axis=None, kind="stable")[:KL_TERMS]
    pos = np.stack(np.unravel_index(order, prod.shape), axis=1)
    return dict(w1d=np.array(w), a1d=np.array(a), lam1d=np.array(lam),
                evpPos=(pos + 1).astype(np.int32), eigs=prod.ravel()[order], M=KL_TERMS,
                kmax=KL_TERMS)


def _xi(seed, case):
    """Standard-normal KL coefficients per class."""
    g = np.random.default_rng(seed)
    return [g.standard_normal((n, KL_TERMS)) for n in _counts(case)]


def _hexes(seed, n):
    """n hexahedra with jittered corners and their lognormal moduli."""
    g = np.random.default_rng(seed)
    corners = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0],
                        [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]], float)
    xyz = g.random((n, 1, 3)) + 0.1 * (corners + g.uniform(-0.15, 0.15, (n, 8, 3)))
    return xyz, MEAN_E * np.exp(0.3 * g.standard_normal(n))


@functools.lru_cache(maxsize=1)
def _context():
    return msa.Context(0)


def _acceleration(case):
    return msa.sinusoidal_history(0.05, 1e-4, 0.05, 1.0, case["steps"])


def prepare(case, seed):
    ctx = _context()
    if case["kind"] == "ke":
        xyz, E = _hexes(seed, case["elements"])
        return {"case": case, "provider": msa.ElementStructuralStiffnessProvider(ctx),
                "xyz": xyz, "E": E}
    boxes, counts = _boxes(case), _counts(case)
    models = [msa.cantilever(*b, *_lengths(b), load=LOAD) for b in boxes]
    meshes = [msa.Mesh(ctx, m.xyz, m.conn, m.dof, m.n_free) for m in models]
    kind = case["kind"]
    precision = PRECISION[case.get("precision", "fp64")]
    b = msa.Batch(ctx, meshes, counts, precision)
    precond = PRECOND[case.get("precond", "jacobi")]
    if precond != msa.MSA_PRECOND_JACOBI:
        b.set_preconditioner(precond)
    if kind == "direct":
        b.set_solver(msa.MSA_SOLVER_DIRECT)
    xi = _xi(seed, case)
    for c, m in enumerate(models):
        b.set_kl(c, _kl_table(_lengths(boxes[c])), m.domain, MEAN_E, case["cov"])
        if kind != "newmark":
            b.set_rhs(c, m.f)
    state = {"case": case, "batch": b, "meshes": meshes, "xi": xi, "counts": counts}
    if kind == "newmark":
        b.set_dynamics(7.85e-9, case["rayleigh_alpha"], case["rayleigh_beta"], 0.25, 0.5, 1e-4)
        for c, m in enumerate(models):
            b.set_probe(c, m.n_free - 1)
        state["acc"] = _acceleration(case)
    if kind == "results":
        # a solved sample in hand, as an analysis has before it asks for stresses
        b.set_xi(0, xi[0])
        b.run(NU, tol=1e-12, max_it=MAX_IT, graph_iters=12)
    # the program's own arrays of every sample's result
    fields = [np.zeros((n, m.n_free)) for n, m in zip(counts, models)]
    state["out"] = {"u": fields}
    if kind == "newmark":
        state["out"] = {"history": np.zeros((counts[0], case["steps"])), "u": fields[0],
                        "a": fields[0].copy()}
    ctx.synchronize()
    return state


# --------------------------------------------------------------------- run

def _split(o, k):
    """The first k samples' rows, whose exact result is formed, and the rest."""
    return [o[:k], o[k:]] if o.shape[0] > k else [o]


def run(state):
    """One pass; host arrays, as the entry points return them."""
    case = state["case"]
    kind = case["kind"]
    if kind == "ke":
        return state["provider"].Matrix(state["xyz"], state["E"], NU)
    b = state["batch"]
    if kind == "results":
        return b.element_results(0, 0)
    for c, xi in enumerate(state["xi"]):
        b.set_xi(c, xi)
    out, counts = state["out"], state["counts"]
    if kind == "newmark":
        b.eval_kl()
        b.assemble(NU)
        b.newmark(state["acc"], 2, case["tol"], MAX_IT, case["graph_iters"])
        for s in range(counts[0]):
            out["history"][s] = b.history(0, s)
            # the velocity is left out: under this quasi-static load it
            # cancels to nearly zero after every second step
            out["u"][s], _, out["a"][s], _ = b.dynamic_state(0, s)
        return {k: _split(o, 1) for k, o in out.items()}
    b.run(NU, tol=case.get("tol", 1e-10), max_it=MAX_IT, graph_iters=case.get("graph_iters", 0))
    for c, n in enumerate(counts):
        for s in range(n):
            out["u"][c][s] = b.solution(c, s)
    return {"u": [_split(o, EXACT_SAMPLES) for o in out["u"]],
            "status": [b.stats(c)["status"] for c in range(len(counts))]}


# -------------------------------------------------------------------- work

def _nodes(box):
    return box[0] * (box[1] + 1) * (box[2] + 1)  # free nodes


def _products(case, box):
    """Operator products of one solve of a block: PCG iterations (Jacobi
    about 20 per element along x with a random modulus, 12 with multigrid of
    5 products each, 25 with the first sample's factor)."""
    precond = case.get("precond", "jacobi")
    if precond == "multigrid" and all(v % 2 == 0 for v in box):
        return 12 * 5
    if precond == "first_sample":
        return 25
    return 20 * max(box)


def work(case):
    """Inputs read once, outputs written once; a product counts the 27 3x3
    blocks of every free node's row, a factorization n * bandwidth^2."""
    kind = case["kind"]
    if kind == "ke":
        n = case["elements"]
        # 8 Gauss points, upper triangle of B^T D B with its block structure
        return {"bytes": n * (25 + 300) * 8.0, "flops": n * 8 * 300 * 6.0}
    nbytes = flops = 0.0
    for box, n in zip(_boxes(case), _counts(case)):
        nodes, elems = _nodes(box), box[0] * box[1] * box[2]
        if kind == "results":
            nbytes += 8.0 * (3 * nodes + elems + elems * (48 + 48 + 24))
            flops += elems * 8 * 2.0 * (24 * 6 + 6 * 6 + 24 * 6)
            continue
        nbytes += 8.0 * n * (KL_TERMS + 3 * nodes)
        flops += n * elems * (2.0 * KL_TERMS)
        if kind == "direct":
            rows = sorted(v + 1 for v in box)
            flops += n * 3.0 * nodes * (3.0 * rows[0] * rows[1]) ** 2
            continue
        steps = case.get("steps", 1)
        flops += n * steps * _products(case, box) * 486.0 * nodes
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the largest error against `exact` seen over the
    ranges (in brackets); for the iterative solves it follows the stopping
    test, at which two correct solvers may end anywhere below it."""
    kind = case["kind"]
    if kind == "ke":
        return {"rel": 4e-15}   # [9.2e-16]
    if kind == "direct":
        return {"rel": 1e-12}   # [2.1e-13]
    if kind == "results":
        return {"rel": 2e-10}   # [4.5e-11: displacements solved to 1e-12]
    if kind == "newmark":
        return {"rel": 4e-9}    # [5.8e-10, accelerations; steps solved to 1e-8]
    if case["precision"] == "mixed":
        return {"rel": 2e-9}    # [5.3e-10, residual below 1e-9]
    return {"rel": case["tol"]}  # [0.2 x the residual bound of 1e-10]


# ------------------------------------------------------------------- exact

CORNERS = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))
SIGN = 2.0 * np.array(CORNERS) - 1.0


def _gauss_points():
    g = (-GAUSS, GAUSS)
    return [np.array([x, y, z]) for x in g for y in g for z in g]


def _elastic(E):
    """Isotropic 6x6 matrices (xx, yy, zz, xy, yz, zx; engineering shear)."""
    D = np.zeros(np.shape(E) + (6, 6))
    e1 = E / (1.0 + NU)
    lam = e1 * NU / (1.0 - 2.0 * NU)
    for i in range(3):
        for j in range(3):
            D[..., i, j] = lam
        D[..., i, i] += e1
        D[..., 3 + i, 3 + i] = 0.5 * e1
    return D


def _strain_matrices(xyz):
    """B [8, n, 6, 24] and w [8, n] at the Gauss points of n hexahedra."""
    Bs, ws = [], []
    for p in _gauss_points():
        dN = np.empty((8, 3))
        for d in range(3):
            o, q = (d + 1) % 3, (d + 2) % 3
            dN[:, d] = 0.125 * SIGN[:, d] * (1 + SIGN[:, o] * p[o]) * (1 + SIGN[:, q] * p[q])
        J = np.einsum("ad,naj->ndj", dN, xyz)
        G = np.einsum("njd,ad->naj", np.linalg.inv(J), dN)  # dN/dx
        B = np.zeros((xyz.shape[0], 6, 24))
        for i in range(3):
            B[:, i, i::3] = G[:, :, i]
        for r, (i, j) in enumerate(((0, 1), (1, 2), (2, 0))):
            B[:, 3 + r, i::3] = G[:, :, j]
            B[:, 3 + r, j::3] = G[:, :, i]
        Bs.append(B)
        ws.append(np.linalg.det(J))
    return np.array(Bs), np.array(ws)


def _unit_matrices(h):
    """Unit-modulus stiffness and unit-density mass of a cubic cell."""
    xyz = (np.array(CORNERS, float) * h)[None]
    B, w = _strain_matrices(xyz)
    D = _elastic(np.float64(1.0))
    K = np.einsum("gnri,rs,gnsj,gn->ij", B, D, B, w)
    M = np.zeros((24, 24))
    for p, wg in zip(_gauss_points(), w[:, 0]):
        N = np.prod(0.5 * (1.0 + SIGN * p), axis=1)
        for d in range(3):
            M[d::3, d::3] += wg * np.outer(N, N)
    return K, M


def _field(box, xi, cov):
    """Lognormal modulus [samples, z, y, x] at the cell centres."""
    t, L = _kl_table(_lengths(box)), _lengths(box)
    sigma = math.sqrt(math.log(cov * cov + 1.0))
    c = [(np.arange(n) + 0.5) * (l / n) - l / 2 for n, l in zip(box, L)]
    f = []
    for d in range(3):
        idx = t["evpPos"][:, d]
        arg = t["w1d"][d][idx - 1][:, None] * c[d][None, :]
        f.append(t["a1d"][d][idx - 1][:, None] *
                 np.where(idx[:, None] % 2 == 0, np.sin(arg), np.cos(arg)))
    phi = (sigma * np.sqrt(t["eigs"]))[:, None, None, None] * \
        f[2][:, :, None, None] * f[1][:, None, :, None] * f[0][:, None, None, :]
    g = np.tensordot(xi, phi, axes=1)
    return np.exp(math.log(MEAN_E) - 0.5 * sigma ** 2 + g)


class _Block:
    """The operator cK E K + cM M of a clamped block in 64-bit torch, node
    vectors [samples, z, y, x, 3] with the held face x = 0 kept at zero."""

    def __init__(self, box, E):
        self.box = box
        self.E = torch.as_tensor(E, dtype=torch.float64).to(_device())
        K, M = _unit_matrices(_lengths(box)[0] / box[0])
        self.K = torch.as_tensor(K).to(_device())
        self.M = torch.as_tensor(M).to(_device())
        self.shape = (self.E.shape[0], box[2] + 1, box[1] + 1, box[0] + 1, 3)

    def _parts(self, U):
        nx, ny, nz = self.box
        return [U[:, dz:dz + nz, dy:dy + ny, dx:dx + nx] for dx, dy, dz in CORNERS]

    def apply(self, U, cK, cM):
        G = torch.stack(self._parts(U), dim=4).flatten(4)
        F = (G @ self.K) * (cK * self.E)[..., None]
        if cM:
            F = F + G @ (cM * self.M)
        F = F.unflatten(4, (8, 3))
        out = torch.zeros(self.shape, dtype=torch.float64, device=U.device)
        for a, part in enumerate(self._parts(out)):
            part += F[..., a, :]
        out[:, :, :, 0] = 0
        return out

    def diagonal(self, cK, cM):
        d = (cK * self.E)[..., None] * torch.diagonal(self.K) + cM * torch.diagonal(self.M)
        d = d.unflatten(4, (8, 3))
        out = torch.zeros(self.shape, dtype=torch.float64, device=d.device)
        for a, part in enumerate(self._parts(out)):
            part += d[..., a, :]
        return out

    def load(self):
        f = torch.zeros(self.shape, dtype=torch.float64, device=self.E.device)
        f[:, :, :, -1, 2] = LOAD / ((self.box[1] + 1) * (self.box[2] + 1))
        return f

    def solve(self, f, cK=1.0, cM=0.0, u=None):
        """Jacobi-CG, restarted on the true residual until it stagnates."""
        dot = lambda x, y: (x * y).sum((1, 2, 3, 4), keepdim=True)
        d = self.diagonal(cK, cM)
        u = torch.zeros_like(f) if u is None else u
        target = 1e-28 * dot(f, f)
        for _ in range(2):
            r = f - self.apply(u, cK, cM)
            r[:, :, :, 0] = 0
            x = torch.zeros_like(f)
            z = r / d
            p, rz = z.clone(), dot(r, z)
            for it in range(MAX_IT):
                q = self.apply(p, cK, cM)
                pq = dot(p, q)
                alpha = torch.where(pq > 0, rz / pq, 0.0)
                x += alpha * p
                r -= alpha * q
                z = r / d
                new = dot(r, z)
                p = z + torch.where(rz > 0, new / rz, 0.0) * p
                rz = new
                if it % 25 == 24 and bool((dot(r, r) <= target).all()):
                    break
            u = u + x
        return u

    def vectors(self, U):
        return U[:, :, :, 1:].reshape(U.shape[0], -1).cpu().numpy()


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _exact_newmark(case, box, xi):
    blk = _Block(box, _field(box, xi, case["cov"]))
    rho, aR, bR = 7.85e-9, case["rayleigh_alpha"], case["rayleigh_beta"]
    alpha, delta, dt = 0.25, 0.5, 1e-4
    a0, a1, a2 = 1 / (alpha * dt * dt), delta / (alpha * dt), 1 / (alpha * dt)
    a3, a4 = 1 / (2 * alpha) - 1, delta / alpha - 1
    a5, a6, a7 = dt * 0.5 * (delta / alpha - 2), dt * (1 - delta), delta * dt
    ones = torch.zeros(blk.shape, dtype=torch.float64, device=blk.E.device)
    ones[..., 2] = 1.0
    base = blk.apply(ones, 0.0, rho)
    u, v, a = (torch.zeros_like(base) for _ in range(3))
    hist = []
    for acc in _acceleration(case):
        wm = a0 * u + a2 * v + a3 * a
        wc = a1 * u + a4 * v + a5 * a
        rhs = float(acc) * base + blk.apply(wm, 0.0, rho) + blk.apply(wc, bR, aR * rho)
        new = blk.solve(rhs, 1.0 + a1 * bR, (a0 + a1 * aR) * rho, u)
        acc_new = a0 * (new - u) - a2 * v - a3 * a
        v = v + a6 * a + a7 * acc_new
        u, a = new, acc_new
        hist.append(u[:, -1, -1, -1, 2].cpu().numpy())
    out = {"history": np.array(hist).T, "u": blk.vectors(u), "a": blk.vectors(a)}
    rest = [None] if _counts(case)[0] > len(xi) else []
    return {k: [o] + rest for k, o in out.items()}


def _exact_results(box, E, u):
    """Strains, stresses and forces of one sample from its displacements."""
    blk = _Block(box, E)
    full = torch.zeros(blk.shape, dtype=torch.float64, device=blk.E.device)
    full[0] = u
    Ue = torch.stack(blk._parts(full), dim=4).flatten(4)[0].reshape(-1, 24).cpu().numpy()
    h = _lengths(box)[0] / box[0]
    B, w = _strain_matrices((np.array(CORNERS, float) * h)[None])
    eps = np.einsum("gri,ei->egr", B[:, 0], Ue)
    sig = np.einsum("rs,egs->egr", _elastic(np.float64(1.0)), eps) * E.reshape(-1)[:, None, None]
    force = np.einsum("gri,egr,g->ei", B[:, 0], sig, w[:, 0])
    return eps, sig, force


def exact(case, seed):
    kind = case["kind"]
    if kind == "ke":
        xyz, E = _hexes(seed, case["elements"])
        B, w = _strain_matrices(xyz)
        K = np.zeros((len(E), 24, 24))
        for g in range(8):
            K += np.einsum("nri,nrs,nsj->nij", B[g], _elastic(E) * w[g][:, None, None], B[g],
                           optimize=True)
        i, j = np.triu_indices(24)
        return K[:, i, j]
    xi = _xi(seed, case)
    boxes, counts = _boxes(case), _counts(case)
    if kind == "newmark":
        return _exact_newmark(case, boxes[0], xi[0][:1])
    out = []
    for box, n, x in zip(boxes, counts, xi):
        k = min(n, EXACT_SAMPLES)
        E = _field(box, x[:k], case["cov"])
        blk = _Block(box, E)
        u = blk.solve(blk.load())
        if kind == "results":
            return _exact_results(box, E, u[0])
        out.append([blk.vectors(u)] + ([None] if n > k else []))
    return {"u": out, "status": [np.zeros(n, np.int32) for n in counts]}
