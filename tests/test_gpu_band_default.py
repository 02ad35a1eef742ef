"""The FP64 band solver where a cell is not positive definite.  With -A for A
the system changes sign: the same bases and M times -1, from pivots that are
all negative.  1e-12 relative: both are one LDL^T without pivoting of the same
numbers (n 2^-53 cond < 1e-12 for these cells)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(verts, dim, l, coef, **kw):
    from msfec_amd import QBasisBatch
    with QBasisBatch(verts, dim=dim, n_refine_local=l, rhs_const=1.0, solver=0, **kw) as qb:
        qb.set_coefficient(coef)
        qb.run()
        return (qb.get_global_element_matrix(), qb.get_basis(), qb.get_cell_status())


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("dim,l,tensor", [(2, 1, False), (2, 4, False), (2, 5, False), (2, 3, True),
                                          (3, 1, False), (3, 2, True), (3, 3, False), (3, 3, True)])
def test_not_positive_definite(oracle_mod, dim, l, tensor):
    print(f"case band default dim={dim} l={l} tensor={tensor}", flush=True)
    from msfec_amd import _lib as L
    from test_gpu_parity import random_boxes, tol
    rng = np.random.default_rng(10 * dim + l)
    nf, n = (1 << l) ** dim, 5
    verts = random_boxes(rng, dim, n)
    verts[1] = verts[3] = verts[0]
    if tensor:
        B = rng.standard_normal((n, nf, 1 << dim, dim, dim))
        A = np.einsum("...ij,...kj->...ik", B, B) + 0.5 * np.eye(dim)
        i, j = np.triu_indices(dim)
        coef = np.ascontiguousarray(A[..., i, j])
    else:
        coef = np.exp(rng.standard_normal((n, nf)))
    coef[1] = -coef[0]
    coef[2, nf // 2] = np.nan
    coef[3] = coef[0]
    kw = dict(coef_mode=1 if tensor else 0)
    M, P, st = run(verts, dim, l, coef, **kw)
    assert st.tolist() == [L.CELL_OK, L.CELL_NOT_SPD, L.CELL_NONFINITE, L.CELL_OK, L.CELL_OK]
    assert rel(-M[1], M[0]) < 1e-12 and rel(P[1], P[0]) < 1e-12
    assert np.array_equal(M[3], M[0]) and np.array_equal(P[3], P[0])
    o = oracle_mod.basis_batch(oracle_mod.make_problem(dim, l, rhs_const=1.0, **kw), verts[4:],
                               coef=coef[4:], solver=oracle_mod.SOLVER_DIRECT, n_threads=2)
    # the oracle takes the sides of each fine cell from its own vertices, the
    # kernels one difference per coarse cell: eps |x| / h per side, 2^l more
    # than the factorisation's bound; the tolerance of the parity tests
    assert rel(M[4:], o["M"]) < tol(0) and rel(P[4:], o["Psi"]) < tol(0)


def test_rounding_of_the_pivots():
    """The matrix-core kernel scales by inverse roots, the one-pivot kernel
    (reached with -A, the same bases) divides: the mean error of the bases of
    64 cells of 32^2, against a solution refined with residuals in extended
    precision, is the same to a tenth.  (With inverse roots off by three
    roundings it is a fifth larger.)"""
    print("case band default rounding", flush=True)
    import scipy.sparse as sp
    import scipy.sparse.linalg as spl
    from msfec_amd import fields as F
    nc, N = 8, 32
    n, S = nc * nc, N + 1
    coef = np.exp(np.random.default_rng(71).standard_normal((n, N * N)))
    verts = F.coarse_vertices(2, nc)
    _, P, st = run(verts, 2, 5, coef)
    _, Q, sq = run(verts, 2, 5, -coef)
    assert (st == 0).all() and (sq != 0).all()
    Ke = np.array([[4, -1, -1, -2], [-1, 4, -2, -1], [-1, -2, 4, -1], [-2, -1, -1, 4]])
    i = np.arange(N * N)
    node = (i // N * S + i % N)[:, None] + np.array([0, 1, S, S + 1])
    x, y = np.arange(S * S) % S, np.arange(S * S) // S
    free = (x > 0) & (x < N) & (y > 0) & (y < N)
    X, Y = x / N, y / N
    g = np.stack([(1 - X) * (1 - Y), X * (1 - Y), (1 - X) * Y, X * Y]).astype(np.longdouble)
    g[:, free] = 0
    e = [0.0, 0.0]
    for c in range(n):
        def apply(v):
            out = np.zeros_like(v)
            np.add.at(out.T, node, ((v[:, node] @ Ke) / np.longdouble(6) * coef[c][:, None]).transpose(1, 2, 0))
            return out
        K = sp.coo_matrix(((coef[c][:, None, None] * Ke / 6.0).ravel(),
                           (np.repeat(node, 4, 1).ravel(), np.tile(node, (1, 4)).ravel())),
                          shape=(S * S,) * 2).tocsc()[free][:, free]
        lu = spl.splu(K)
        psi = g.copy()
        for _ in range(4):
            psi[:, free] -= lu.solve(apply(psi)[:, free].T.astype(float)).T
        for k, B in enumerate((P, Q)):
            e[k] += float(np.linalg.norm(B[c] - psi) / np.linalg.norm(psi)) / n
    print("matrix cores %.2e, divisions %.2e" % tuple(e), flush=True)
    assert e[0] <= 1.1 * e[1], e
