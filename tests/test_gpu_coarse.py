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
