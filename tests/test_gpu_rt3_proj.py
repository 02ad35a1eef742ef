"""The 3-D RT_DQ fluxes by projected conjugate gradients, on every grid size of
the kernels and on both sides of the contrast above which the curl-curl solver
takes a cell."""
import numpy as np
import pytest

from test_gpu_nrt import boxes, rand_coefs

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def run(verts, l, ainv, f=None, **kw):
    from msfec_amd import RTDQ3BasisBatch
    with RTDQ3BasisBatch(verts, n_refine_local=l, **kw) as rb:
        rb.set_coefficients(ainv, f)
        rb.run()
        return (rb.get_global_element_matrix(), rb.get_global_element_rhs(), rb.get_basis(),
                rb.get_cell_status(), rb.get_iterations())


@pytest.mark.parametrize("l,n", [(1, 17), (2, 9), (3, 3)])
def test_contrasts_in_one_batch(oracle_mod, l, n):
    """Stretched boxes with rotated tensors, cell c scaled by lognormal factors
    of deviation 0, 1, 2, .. 6 in turn (contrast 1e1 to beyond 1e8: the last
    ones are left to the curl-curl solver).  Both solvers stop at 1e-13 of a
    residual, which leaves at most the square root of the contrast times as
    much in the flux: ten times that, and never more than 1e-9.  M is of second
    order in it: 1e-13 (2e-15 measured)."""
    print(f"case rt3 contrasts l={l} n={n}", flush=True)
    rng = np.random.default_rng(5000 + l)
    verts = boxes(rng, n)
    ainv, _, _, _ = rand_coefs(rng, n, l, reaction=False, load=False)
    f = rng.normal(size=(n, 8 ** l, 8))
    dev = np.arange(n) % 7
    ainv = ainv * np.exp(dev[:, None, None, None] * rng.normal(size=ainv.shape[:2] + (1, 1)))
    M, b, S, st, its = run(verts, l, ainv, f)
    assert (st == 0).all(), st
    for c in range(n):
        Mo, bo, So, sto = oracle_mod.rt3_basis_cell(l, verts[c], ainv[c], f[c])
        assert sto == 0
        trace = ainv[c][..., [0, 3, 5]].sum(-1)
        tol = min(1e-12 * np.sqrt(trace.max() / trace.min()), 1e-9)
        es = max(rel(S[c, i], So[i]) for i in range(6))
        print(f"cell {c} deviation {dev[c]}: {es:.1e} {rel(M[c], Mo):.1e} its {its[c].max()}", flush=True)
        assert es <= tol and rel(M[c], Mo) <= 1e-13 and rel(b[c], bo) <= 1e-12


@pytest.mark.parametrize("l", [2, 3, 4])
def test_general_cells_do_not_disturb_others(l):
    """Cells that go to the curl-curl solver (indefinite, NaN, huge contrast)
    between cells that do not: the latter come out bit for bit as without
    them."""
    print(f"case rt3 neighbours of general cells l={l}", flush=True)
    rng = np.random.default_rng(5100 + l)
    n = 10
    verts = boxes(rng, n)
    ainv, _, _, _ = rand_coefs(rng, n, l, reaction=False, load=False)
    good = run(verts, l, ainv, max_iter=300)
    ainv[1] = -ainv[1]
    ainv[4, 3, 2, 0] = np.nan
    ainv[7, ::2] *= 1e9
    ainv[9, 0, 0, 3] = -1e-3
    got = run(verts, l, ainv, max_iter=300)
    assert got[3][1] != 0 and got[3][4] != 0
    for c in (0, 2, 3, 5, 6, 8):
        assert got[3][c] == 0
        for k in range(3):
            np.testing.assert_array_equal(got[k][c], good[k][c])


@pytest.mark.parametrize("l,n", [(3, 300), (4, 50)])
def test_equal_cells_come_out_equal(l, n):
    """More workgroups than the card runs at once, all with the same data, over
    several passes: every cell bit for bit the same (the waves of a workgroup
    share their flux lattice, so the order in which they run must not show)."""
    print(f"case rt3 equal cells l={l} n={n}", flush=True)
    from msfec_amd import RTDQ3BasisBatch
    rng = np.random.default_rng(5200 + l)
    verts = np.repeat(boxes(rng, 1), n, 0)
    ainv, _, _, _ = rand_coefs(rng, 1, l, reaction=False, load=False)
    one = run(verts[:1], l, ainv)
    assert one[3][0] == 0
    with RTDQ3BasisBatch(verts, n_refine_local=l) as rb:
        rb.set_coefficients(np.repeat(ainv, n, 0))
        for _ in range(3):
            rb.run()
            got = (rb.get_global_element_matrix(), rb.get_global_element_rhs(), rb.get_basis(),
                   rb.get_cell_status(), rb.get_iterations())
            for a, b in zip(got, one):
                np.testing.assert_array_equal(a, np.broadcast_to(b, a.shape))


@pytest.mark.parametrize("l", [1, 2, 3, 4])
def test_units_of_the_coefficient(l):
    """A^-1 in other units, from 2^-320 to 2^330 (about 1e-96 and 1e99): the
    same fluxes and iterations bit for bit, the flux block of M scaled."""
    print(f"case rt3 units l={l}", flush=True)
    rng = np.random.default_rng(5300 + l)
    n = 3
    verts = boxes(rng, n)
    ainv = np.zeros((n, 8 ** l, 8, 6))
    ainv[..., [0, 3, 5]] = np.exp(0.5 * rng.normal(size=(n, 8 ** l, 8, 3)))
    ainv[..., 1] = 0.1 * ainv[..., 0]
    want = run(verts, l, ainv)
    assert (want[3] == 0).all()
    for e in (-320, -100, 100, 330):
        got = run(verts, l, ainv * 2.0 ** e, max_iter=1000)
        assert (got[3] == 0).all(), (e, got[3], got[4].max())
        np.testing.assert_array_equal(got[2], want[2])
        np.testing.assert_array_equal(got[4], want[4])
        np.testing.assert_array_equal(got[0][:, :6, :6], want[0][:, :6, :6] * 2.0 ** e)


@pytest.mark.parametrize("l", [1, 2, 3, 4])
@pytest.mark.parametrize("dev", [0.3, 1.0, 1.5, 2.0])
def test_balance_of_every_fine_cell(l, dev):
    """The net outflow of a fine cell is -+1/M^3, to the rounding of its 6
    fluxes and of their sum here (each at most half a unit in the last place
    of the largest flux): 6 eps of it, whatever the iterations."""
    print(f"case rt3 balance l={l} deviation={dev}", flush=True)
    rng = np.random.default_rng(5400 + l)
    n, m = 4, 1 << l
    ainv = np.zeros((n, m ** 3, 8, 6))
    ainv[..., [0, 3, 5]] = np.exp(dev * rng.normal(size=(n, m ** 3, 1, 1)))
    _, _, S, st, _ = run(boxes(rng, n), l, ainv)
    assert (st == 0).all()
    x, y, z = np.split(S, 3, -1)
    x = np.diff(x.reshape(n, 6, m, m, m + 1), axis=4)
    y = np.diff(y.reshape(n, 6, m, m + 1, m), axis=3)
    z = np.diff(z.reshape(n, 6, m + 1, m, m), axis=2)
    want = np.array([-1.0, 1, -1, 1, -1, 1])[None, :, None, None, None] / m ** 3
    off = np.abs(x + y + z - want).max((2, 3, 4)) / np.abs(S).max(2)
    assert off.max() <= 6 * np.finfo(float).eps, off.max() / np.finfo(float).eps


def test_default_stop(oracle_mod):
    """8 cells of 8^3 with the oscillatory tensor of the reference example: the
    mean error of the fluxes at the default rtol is at most what the curl-curl
    solver's |r| <= 1e-13 |b| leaves there (1.7e-14 in the 2-norm; the oracle
    is refined to rounding)."""
    print("case rt3 default stop", flush=True)
    from msfec_amd import fields as F
    l, N, n = 3, 8, 8
    verts = F.coarse_vertices(3, 2)
    i = np.arange(N ** 3)
    cell = np.stack([i % N, i // N % N, i // (N * N)], -1)
    q = np.arange(8)
    gp = np.array([0.5 - 0.5 / np.sqrt(3), 0.5 + 0.5 / np.sqrt(3)])
    pt = (cell[:, None] + gp[np.stack([q & 1, q >> 1 & 1, q >> 2], -1)]) / N
    x = verts[:, 0][:, None, None] + pt * 0.5
    phase = np.array([0.1, 0.45, 0.8])
    d = 1.0 / (1.0 - 0.9 * np.sin(2 * np.pi * (np.array([17.0, 16.0, 15.0]) * x + phase)))
    R = F._euler_rotation()
    ainv = np.stack([(R[a] * R[b] * d).sum(-1)
                     for a, b in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))], -1)
    _, _, S, st, its = run(verts, l, ainv)
    assert (st == 0).all()
    e = [np.linalg.norm(S[c] - So) / np.linalg.norm(So)
         for c in range(n) for So in [oracle_mod.rt3_basis_cell(l, verts[c], ainv[c], None)[2]]]
    print("mean %.2e max %.2e its %d" % (np.mean(e), np.max(e), its.max()), flush=True)
    assert np.mean(e) <= 1.7e-14


@pytest.mark.parametrize("l", [1, 2, 3])
def test_smallest_rtol(l):
    """An rtol of 1e-15 is reached at every size (the stop at half of rtol does
    not go below what rounding allows)."""
    print(f"case rt3 smallest rtol l={l}", flush=True)
    rng = np.random.default_rng(5500 + l)
    n = 9
    ainv, _, _, _ = rand_coefs(rng, n, l, reaction=False, load=False)
    _, _, _, st, its = run(boxes(rng, n), l, ainv, rtol=1e-15, max_iter=1000)
    assert (st == 0).all(), (st, its.max())
