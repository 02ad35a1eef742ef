"""3-D Q1 bases by CG on assembled rows (tensors or loads at the Gauss points)
at every grid size of the kernels: M = 2, 4, 8 and 16 nodes a column, with one
and with several cells per group of 8 workgroups, against the oracle's direct
solve.  1e-10 relative, the tolerance of the CG tests (it stops at 1e-13 of
the residual)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CG, TENSOR, SCALAR = 3, 1, 0


def rel(a, b):
    n = a.shape[0]
    num = np.linalg.norm((a - b).reshape(n, -1), axis=1)
    return float(np.max(num / np.linalg.norm(b.reshape(n, -1), axis=1)))


def problem(rng, n, l, coef_mode, rhs_mode, reaction_mode):
    from test_gpu_parity import random_boxes
    nf = 8 ** l
    verts = random_boxes(rng, 3, n)
    if coef_mode == TENSOR:
        B = rng.standard_normal((n, nf, 8, 3, 3))
        A = np.einsum("...ij,...kj->...ik", B, B) + 0.5 * np.eye(3)
        coef = np.stack([A[..., 0, 0], A[..., 0, 1], A[..., 0, 2], A[..., 1, 1], A[..., 1, 2],
                         A[..., 2, 2]], -1)
    else:
        coef = np.exp(rng.standard_normal((n, nf)))
    kw = dict(coef_mode=coef_mode, rhs_mode=rhs_mode, rhs_const=0.7, reaction_mode=reaction_mode,
              reaction_const=30.0 if reaction_mode == 1 else 0.0)
    f = None if rhs_mode == 0 else rng.standard_normal((n, nf) if rhs_mode == 1 else (n, nf, 8))
    r = None if reaction_mode != 2 else 50.0 * rng.random((n, nf))
    return verts, coef, f, r, kw


@pytest.mark.parametrize("l,n,coef_mode,rhs_mode,reaction_mode", [
    (1, 3, TENSOR, 2, 0), (1, 9, SCALAR, 2, 2), (2, 11, TENSOR, 0, 1), (2, 4, SCALAR, 2, 0),
    (3, 9, TENSOR, 1, 2), (3, 2, SCALAR, 2, 1), (4, 2, TENSOR, 2, 2), (4, 1, SCALAR, 2, 0)])
def test_matches_oracle(oracle_mod, l, n, coef_mode, rhs_mode, reaction_mode):
    print(f"case q1t l={l} n={n} {coef_mode} {rhs_mode} {reaction_mode}", flush=True)
    from msfec_amd import QBasisBatch
    rng = np.random.default_rng(4000 + 10 * l + n)
    verts, coef, f, r, kw = problem(rng, n, l, coef_mode, rhs_mode, reaction_mode)
    with QBasisBatch(verts, dim=3, n_refine_local=l, solver=CG, **kw) as qb:
        qb.set_coefficient(coef)
        if f is not None:
            qb.set_rhs(f)
        if r is not None:
            qb.set_reaction(r)
        qb.run()
        M, b, P, st = (qb.get_global_element_matrix(), qb.get_global_element_rhs(), qb.get_basis(),
                       qb.get_cell_status())
        it = qb.cg_iterations()
    assert (st == 0).all() and (it > 0).all()
    if reaction_mode == 0:  # the last basis follows from the others
        assert (it[:, 7] == it[:, :7].max(axis=1)).all()
    o = oracle_mod.basis_batch(oracle_mod.make_problem(3, l, **kw), verts, coef=coef, f=f, reaction=r,
                               solver=oracle_mod.SOLVER_DIRECT, n_threads=8)
    assert rel(M, o["M"]) < 1e-10 and rel(P, o["Psi"]) < 1e-10
    assert rel(b, o["b"]) < 1e-10


def test_limit_breakdown_and_nonfinite():
    """An iteration limit, a negative definite tensor and a NaN flag their own
    cells only."""
    print("case q1t flags", flush=True)
    from msfec_amd import QBasisBatch, _lib as L
    rng = np.random.default_rng(4100)
    verts, coef, f, r, kw = problem(rng, 10, 3, TENSOR, 0, 0)
    coef[3] = -coef[3]
    coef[8, 17, 5, 0] = np.nan
    with QBasisBatch(verts, dim=3, n_refine_local=3, solver=CG, **kw) as qb:
        qb.set_coefficient(coef)
        qb.run()
        st = qb.get_cell_status()
    assert st[3] == L.CELL_NOT_SPD and st[8] in (L.CELL_NOT_SPD, L.CELL_NONFINITE)
    assert (np.delete(st, [3, 8]) == 0).all()
    with QBasisBatch(verts[:2], dim=3, n_refine_local=3, solver=CG, cg_max_iter=4, **kw) as qb:
        qb.set_coefficient(coef[:2])
        qb.run()
        assert (qb.get_cell_status() == L.CELL_NOT_CONVERGED).all()
        assert (qb.cg_iterations() == 4).all()
