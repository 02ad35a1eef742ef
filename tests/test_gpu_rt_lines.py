"""2-D RT_DQ at l = 4 and 5, where the bases come from the reduction by lines
of nodes: against the oracle at the oracle's sizes (l = 4) and, at l = 5,
against the same cell under a rotation by 180 degrees, which reverses the
order of elimination; and cells that are not positive definite next to ones
that are.  With -a the reduced system changes sign: the same fluxes, the flux
block of M times -1.  1e-11, the bound of two direct solves of conditioning
max(a) / min(a) (the tolerance of the other RT_DQ tests)."""
import numpy as np
import pytest

from test_gpu_rt import TOL_M, TOL_S, boxes, compare, run_gpu

pytestmark = pytest.mark.gpu


def coefficient(rng, n, l, tensor):
    nf = 4 ** l
    if not tensor:
        return np.exp(rng.normal(size=(n, nf)))
    B = rng.normal(size=(n, nf, 4, 2, 2))
    A = np.einsum("...ij,...kj->...ik", B, B) + 0.2 * np.eye(2)
    return np.ascontiguousarray(np.stack([A[..., 0, 0], A[..., 0, 1], A[..., 1, 1]], -1))


@pytest.mark.parametrize("l,n,tensor", [(4, 1, False), (4, 9, True), (5, 1, True), (5, 5, False)])
def test_lines(oracle_mod, l, n, tensor):
    print(f"case rt lines l={l} n={n} tensor={tensor}", flush=True)
    rng = np.random.default_rng(900 + 10 * l + n)
    verts, a = boxes(rng, n), coefficient(rng, n, l, tensor)
    M, b, S, st = run_gpu(verts, l, a, 1.0, tensor)
    assert (st == 0).all()
    if l == 4 and not tensor:
        compare(M, b, S, oracle_mod.rt_basis_batch(l, verts, a, np.ones_like(a)))
    # rotated: cell (i, j) <-> (m-1-i, m-1-j), bases 0 <-> 1 and 2 <-> 3 with
    # the sign of the normal, Gauss points 0 <-> 3 and 1 <-> 2
    ar = np.ascontiguousarray(a[:, ::-1][:, :, ::-1] if tensor else a[:, ::-1])
    Mr, _, _, sr = run_gpu(verts, l, ar, 1.0, tensor)
    p = [1, 0, 3, 2]
    assert (sr == 0).all()
    for c in range(n):
        assert np.abs(Mr[c][:4, :4][np.ix_(p, p)] - M[c, :4, :4]).max() <= TOL_M * np.abs(M[c, :4, :4]).max()


@pytest.mark.parametrize("l,tensor", [(4, False), (4, True), (5, False)])
def test_not_positive_definite(l, tensor):
    print(f"case rt lines indefinite l={l} tensor={tensor}", flush=True)
    rng = np.random.default_rng(950 + l)
    verts, a = boxes(rng, 5), coefficient(rng, 5, l, tensor)
    verts[1] = verts[3] = verts[0]
    a[1] = -a[0]
    a[2, 4 ** l // 2] = np.nan
    a[3] = a[0]
    M, _, S, st = run_gpu(verts, l, a, 1.0, tensor)
    assert (st[[0, 1, 3, 4]] == 0).all() and st[2] != 0
    assert np.abs(S[1] - S[0]).max() <= TOL_S * np.abs(S[0]).max()
    assert np.abs(M[1, :4, :4] + M[0, :4, :4]).max() <= TOL_M * np.abs(M[0, :4, :4]).max()
    assert np.array_equal(S[3], S[0]) and np.isfinite(S[4]).all()


@pytest.mark.parametrize("l,n", [(4, 1536), (4, 1537), (5, 640), (5, 641)])
def test_sides_of_the_rule(l, n):
    """The same cells by lines and, one cell more, by the band solve."""
    print(f"case rt lines rule l={l} n={n}", flush=True)
    rng = np.random.default_rng(970 + l)
    verts, a = boxes(rng, 4), coefficient(rng, 4, l, False)
    pick = np.arange(n) % 4
    M, _, S, st = run_gpu(verts[pick], l, a[pick], 1.0)
    few, _, Sf, _ = run_gpu(verts, l, a, 1.0)
    assert (st == 0).all()
    for c in (0, 1, 2, 3, n - 1):
        assert np.abs(S[c] - Sf[c % 4]).max() <= TOL_S * np.abs(Sf[c % 4]).max()
        assert np.abs(M[c, :4, :4] - few[c % 4, :4, :4]).max() <= TOL_M * np.abs(few[c % 4, :4, :4]).max()
