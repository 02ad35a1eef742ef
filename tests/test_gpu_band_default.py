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
