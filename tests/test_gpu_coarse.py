"""The coarse solve at the sizes where its kernel changes: one node, one wave,
one node per thread up to 1024, four per thread up to 4096, and beyond.  The
residual b - K u of the assembled problem, formed here from the element
matrices, is at most the tolerance of the iteration plus the gap between the
recursive and the true residual, eps |K| |u| per iteration (every update of r
and of u rounds once)."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,nc", [(2, 2), (2, 9), (2, 10), (2, 33), (2, 34), (2, 65), (2, 66),
                                    (3, 2), (3, 5), (3, 11), (3, 12), (3, 17), (3, 18)])
def test_coarse_residual(dim, nc):
    print(f"case coarse dim={dim} nc={nc}", flush=True)
    from msfec_amd import QBasisBatch
    from msfec_amd import fields as F
    rng = np.random.default_rng(7 * nc + dim)
    n, nv, S = nc ** dim, 1 << dim, nc + 1
    with QBasisBatch(F.coarse_vertices(dim, nc), dim=dim, n_refine_local=1, rhs_const=1.0) as qb:
        qb.set_coefficient(np.exp(rng.standard_normal((n, nv))))
        qb.run()
        M, b = qb.get_global_element_matrix(), qb.get_global_element_rhs()
        u, w, it, res = qb.coarse_solve(nc, abs_tol=0.0, rel_tol=1e-12)
        if nc > 2:
            with pytest.raises(RuntimeError, match="did not converge"):
                qb.coarse_solve(nc, abs_tol=0.0, rel_tol=1e-12, max_iter=1)
    c = np.stack(np.unravel_index(np.arange(n), (nc,) * dim)[::-1])  # x fastest
    v = np.stack([(np.arange(nv) >> d) & 1 for d in range(dim)])
    node = ((c[:, :, None] + v[:, None, :]) * (S ** np.arange(dim))[:, None, None]).sum(0)
    K = sp.coo_matrix((M.ravel(), (np.repeat(node, nv, 1).ravel(), np.tile(node, (1, nv)).ravel())),
                      shape=(S ** dim,) * 2).tocsr()
    rhs = np.bincount(node.ravel(), b.ravel(), S ** dim)
    x = np.stack(np.unravel_index(np.arange(S ** dim), (S,) * dim))
    free = ((x > 0) & (x < nc)).all(0)
    assert it > 0 and (u[~free] == 0.0).all() and np.array_equal(w, u[node])
    gap = it * np.finfo(float).eps * np.linalg.norm((abs(K) @ abs(u))[free])
    true = np.linalg.norm((rhs - K @ u)[free])
    assert true <= 1e-12 * np.linalg.norm(rhs[free]) + gap, (true, res, gap)
    assert res <= 1e-12 * np.linalg.norm(rhs[free])


@pytest.mark.parametrize("dim,nc", [(2, 9), (2, 34), (2, 66), (2, 115), (3, 5), (3, 12), (3, 18)])
def test_coarse_failures(dim, nc):
    """A load that is not finite, a matrix that is not (the solve fails before
    its first iteration) or that is negative definite (at its first step), and
    a limit of no iterations are errors on every kernel, and leave the handle
    fit for the next solve."""
    print(f"case coarse failures dim={dim} nc={nc}", flush=True)
    from msfec_amd import QBasisBatch, _lib as L
    from msfec_amd import fields as F
    n, nf = nc ** dim, 1 << dim
    coef, f = np.ones((n, nf)), np.ones((n, nf))
    with QBasisBatch(F.coarse_vertices(dim, nc), dim=dim, n_refine_local=1,
                     rhs_mode=L.RHS_CELL) as qb:
        def fails(c, load, **kw):
            qb.set_coefficient(c)
            qb.set_rhs(load)
            qb.run()
            with pytest.raises(RuntimeError, match="did not converge"):
                qb.coarse_solve(nc, abs_tol=0.0, rel_tol=1e-12, **kw)

        for v in (np.nan, np.inf, -np.inf):
            g = f.copy()
            g[n // 2, 0] = v
            fails(coef, g)
        c = coef.copy()
        c[n // 2, 0] = np.nan
        fails(c, f)
        if nc < 100:  # the general kernel takes a negative definite matrix
            fails(-coef, f)
        fails(coef, f, max_iter=0)
        qb.set_coefficient(coef)
        qb.set_rhs(0 * f)
        qb.run()
        u, _, it, res = qb.coarse_solve(nc, abs_tol=0.0, rel_tol=1e-12)
        assert it == 0 and res == 0.0 and (u == 0.0).all()
        qb.set_rhs(f)
        qb.run()
        u, _, it, res = qb.coarse_solve(nc, abs_tol=0.0, rel_tol=1e-12)
        assert it > 0 and u.max() > 0.0


def test_adjoint_failures():
    """The gradient goes by the same solves: a target that is not finite is an
    error inside and does not count on the boundary."""
    print("case adjoint failures", flush=True)
    from msfec_amd import QBasisBatch, _lib as L
    from msfec_amd import fields as F
    nc = 4
    with QBasisBatch(F.coarse_vertices(3, nc), dim=3, n_refine_local=1,
                     solver=L.SOLVER_BAND_FP64_MFMA) as qb:
        qb.set_coefficient(np.ones((nc ** 3, 8)))
        qb.run()
        t = np.zeros((nc + 1,) * 3)
        J, g = qb.adjoint_gradient(nc, t)
        t[0] = np.nan
        Jb, gb = qb.adjoint_gradient(nc, t)
        assert Jb == J and np.array_equal(gb, g)
        t[2, 2, 2] = np.nan
        with pytest.raises(RuntimeError, match="did not converge"):
            qb.adjoint_gradient(nc, t)
