"""Ned_RT without a reaction term: the bases by the exact sequence (the
default path then) against the oracle's direct solves, the general solvers and
closed forms, and the cells that it leaves to the general solvers."""
import numpy as np
import pytest

from test_gpu_nrt import boxes, rand_coefs

pytestmark = pytest.mark.gpu


def run(verts, l, ainv, bq, rq=None, fq=None, **kw):
    from msfec_amd import NedRTBasisBatch
    with NedRTBasisBatch(verts, n_refine_local=l, **kw) as nb:
        nb.set_coefficients(ainv, bq, rq, fq)
        nb.run()
        its = nb.get_iterations() if l > 2 or kw.get("solver") else None
        return (nb.get_global_element_matrix(), nb.get_global_element_rhs(), nb.get_basis(),
                nb.get_cell_status(), its)


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("l,n,load", [(1, 9, True), (2, 17, True), (2, 3, False), (3, 2, True)])
def test_matches_oracle(oracle_mod, l, n, load):
    """Stretched boxes, rotated tensors with a contrast of e^2 between cells;
    1e-11 of each array's largest entry, the tolerance of the direct path
    (the reference solve itself is refined to about 1e-13)."""
    print(f"case nrt sequence l={l} n={n} load={load}", flush=True)
    rng = np.random.default_rng(3000 + l + n)
    verts = boxes(rng, n)
    ainv, bq, _, fq = rand_coefs(rng, n, l, reaction=False, load=load)
    M, b, X, st, its = run(verts, l, ainv, bq, None, fq)
    assert (st == 0).all(), st
    o = oracle_mod.nrt_basis_batch(l, verts, ainv, bq, None, fq, n_threads=8)
    for c in range(n):
        assert rel(M[c], o["M"][c]) <= 1e-11
        for i in range(18):
            assert rel(X[c, i], o["X"][c, i]) <= 1e-11, (c, i)
        assert rel(b[c], o["b"][c]) <= 1e-11 if load else (b[c] == 0).all()
    if its is not None:
        assert (its[:, :12] > 0).all() and (its[:, 12:] == 0).all()


def test_l4_matches_minres():
    """Two cells of 16^3 against MINRES on the full system.  Element matrix and
    load are of second order in the error of either: 1e-12 (2e-15 and 4e-14
    measured).  The bases of MINRES itself are off by up to 1e-9 here (2e-10 to
    4e-10 between its rtol of 1e-14 and 1e-16): 1e-8, the tolerance of its
    tests; those of the sequence must stay within 1e-12 when its rtol goes from
    1e-14 to 1e-17 (3e-14 measured)."""
    print("case nrt sequence l=4", flush=True)
    from msfec_amd import _lib as L
    rng = np.random.default_rng(3104)
    verts = boxes(rng, 2)
    ainv, bq, _, fq = rand_coefs(rng, 2, 4, reaction=False)
    a = run(verts, 4, ainv, bq, None, fq)
    t = run(verts, 4, ainv, bq, None, fq, rtol=1e-17)
    g = run(verts, 4, ainv, bq, None, fq, solver=L.SOLVER_CG)
    assert (a[3] == 0).all() and (t[3] == 0).all() and (g[3] == 0).all()
    for c in range(2):
        assert rel(a[0][c], g[0][c]) <= 1e-12 and rel(a[1][c], g[1][c]) <= 1e-12
        assert max(rel(a[2][c, i], g[2][c, i]) for i in range(18)) <= 1e-8
        assert max(rel(a[2][c, i], t[2][c, i]) for i in range(18)) <= 1e-12


@pytest.mark.parametrize("l", [1, 2, 3])
def test_other_cells_go_to_the_general_solver(l):
    """A negative definite or indefinite A^-1, a Gauss point with B <= 0 or
    NaN: those cells come out as with a zero reaction rate given (which takes
    the whole batch through the general solver), bit for bit; the others do
    not notice."""
    print(f"case nrt sequence fallback l={l}", flush=True)
    rng = np.random.default_rng(3200 + l)
    n = 8
    verts = boxes(rng, n)
    ainv, bq, _, fq = rand_coefs(rng, n, l, reaction=False)
    good = run(verts, l, ainv, bq, None, fq, max_iter=400)
    ainv[1] = -ainv[1]
    ainv[2, 0, 0, 0] = -0.01
    bq[4, 0, 3] = np.nan
    bq[5, 1, 2] = -0.01
    bq[6, 0, 0] = 0.0
    a = run(verts, l, ainv, bq, None, fq, max_iter=400)
    g = run(verts, l, ainv, bq, np.zeros_like(bq), fq, max_iter=400)
    for c in (1, 2, 4, 5, 6):
        assert a[3][c] == g[3][c]
        for k in range(3):
            np.testing.assert_array_equal(a[k][c], g[k][c])
    for c in (0, 3, 7):
        assert a[3][c] == 0
        for k in range(3):
            np.testing.assert_array_equal(a[k][c], good[k][c])


def test_iteration_limit():
    """The limit holds for the conjugate gradients of this path."""
    print("case nrt sequence iteration limit", flush=True)
    from msfec_amd import _lib as L
    rng = np.random.default_rng(3300)
    verts = boxes(rng, 2)
    ainv, bq, _, fq = rand_coefs(rng, 2, 3, reaction=False)
    _, _, _, st, its = run(verts, 3, ainv, bq, None, fq, max_iter=5)
    assert (st == L.CELL_NOT_CONVERGED).all() and (its[:, :12] == 5).all()


@pytest.mark.parametrize("l", [1, 2, 3])
def test_infinite_data(l):
    """An infinite B or A^-1 at one Gauss point, and values of B whose sum over
    a fine cell overflows: flagged, never MSFEC_CELL_OK; a large
    finite value of B passes."""
    print(f"case nrt sequence infinite data l={l}", flush=True)
    rng = np.random.default_rng(3400 + l)
    n = 7
    verts = boxes(rng, n)
    ainv, bq, _, fq = rand_coefs(rng, n, l, reaction=False)
    good = run(verts, l, ainv, bq, None, fq, max_iter=400)
    bq[1, 0, 3] = np.inf
    bq[2, -1, 7] = np.inf
    bq[3, 1, :] = 1e308
    ainv[4, 2, 5, 3] = np.inf
    bq[5, 0, 0] = 1e307
    a = run(verts, l, ainv, bq, None, fq, max_iter=400)
    assert (a[3][[1, 2, 3, 4]] != 0).all(), a[3]
    assert (a[3][[0, 5, 6]] == 0).all(), a[3]
    for c in (0, 6):
        for k in range(3):
            np.testing.assert_array_equal(a[k][c], good[k][c])
