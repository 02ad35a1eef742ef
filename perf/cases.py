"""Timed cases of the multiscale basis library: whole passes through the public
entry points, with the data and the results in device memory.

One pass is what a program does each time its coefficient changes (a new
realisation, a time step, an iteration of an optimiser): hand over the new
coefficient, build the bases of all coarse cells and take what it needs from
them.  That is the element matrices, loads and fine coefficients of the bases
(``want = "basis"``), the coarse solution and its fine reconstruction
(``want = "solution"``) or the gradient of a coarse misfit (``"gradient"``).
The handle, its workspaces and the output buffers are kept between passes.

Kinds (``case["kind"]``), all on the nc^dim cells of the unit cube, each
refined l times:
  q       Q1 basis (QBasisBatch)            uneven  Q1, a level per cell
  ned     2-D Q1 x Nedelec                  rt      2-D Raviart-Thomas x DQ0
  rt3     3-D Raviart-Thomas x DQ0          nrt     3-D Nedelec x Raviart-Thomas

The FP32 + refinement solvers are not timed: they are slower and less precise
than the FP64 ones, so no program has a reason to choose them.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "mpi-msfec_amd"))

from msfec_amd import (NedBasisBatch, NedRTBasisBatch, QBasisBatch, RTDQ3BasisBatch,  # noqa: E402
                       RTDQBasisBatch, UnevenBatch, _lib as L, fields as F)

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
SOLVERS = {"mfma": L.SOLVER_BAND_FP64_MFMA, "default": L.SOLVER_BAND_FP64, "cg": L.SOLVER_CG}


# --------------------------------------------------------------------------- the cases
def listed():
    return [
        # smallest: the 2-D plain method (reaction 1, iid lognormal
        # coefficient) with its coarse solve and reconstruction; launches,
        # waits and the serial coarse CG count
        dict(name="q2_8_l4_solution", kind="q", dim=2, nc=8, l=4, coef="iid", sigma=1.0,
             load="const", reaction="const", solver="mfma", want="solution"),
        # the headline workload: 16^3 cells of 8^3 fine cells, correlated
        # lognormal coefficient (sigma 1.5, correlation length 1/64)
        dict(name="q3_16_l3_basis", kind="q", dim=3, nc=16, l=3, coef="smooth", sigma=1.5,
             load="const", reaction="none", solver="mfma", want="basis"),
        # an odd mesh with what the front ends choose when the caller names no
        # solver, and a load and a reaction rate per fine cell
        dict(name="q3_5_l3_default", kind="q", dim=3, nc=5, l=3, coef="iid", sigma=1.0,
             load="cell", reaction="cell", solver="default", want="basis"),
        # the reference's Q example: 4^3 cells of 16^3, rotated oscillatory
        # tensor and load at the Gauss points, CG
        dict(name="q3_4_l4_tensor", kind="q", dim=3, nc=4, l=4, coef="tensor", sigma=0.9,
             load="qp", reaction="none", solver="cg", want="basis"),
        # backward: gradient of the coarse misfit on the headline mesh
        dict(name="q3_16_l3_gradient", kind="q", dim=3, nc=16, l=3, coef="smooth", sigma=1.5,
             load="const", reaction="none", solver="mfma", want="gradient"),
        # uneven refinement around 410 small stiff inclusions, levels 2, 3, 4
        dict(name="uneven_16", kind="uneven", dim=3, nc=16, inclusions=410, radius=0.02,
             value=1e4),
        # the mixed pairings of the benchmark
        dict(name="ned_32_l4", kind="ned", nc=32, l=4, sigma=1.0),
        dict(name="rt_32_l4", kind="rt", nc=32, l=4, coef="scalar", sigma=1.0),
        # an odd mesh, anisotropic tensors at the Gauss points, the finest level
        dict(name="rt_11_l5_tensor", kind="rt", nc=11, l=5, coef="tensor", sigma=0.9),
        # the reference's 3-D RT_DQ example: 4^3 cells of 16^3
        dict(name="rt3_4_l4", kind="rt3", nc=4, l=4, alpha=0.9),
        # Ned_RT, the dense direct solver on a fine coarse mesh
        dict(name="nrt_16_l2", kind="nrt", nc=16, l=2, alpha=0.9),
        # Ned_RT at the refinement of the reference's examples (MINRES)
        dict(name="nrt_2_l4", kind="nrt", nc=2, l=4, alpha=0.9),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo - 0.49), math.log(hi + 0.49)))))

    kind = rng.choice(["q2", "q3", "q3", "tensor", "gradient", "uneven", "ned", "rt", "rt3", "nrt",
                       "nrt"])
    sigma = round(rng.uniform(0.5, 1.5), 3)
    if kind in ("q2", "q3"):
        dim = 2 if kind == "q2" else 3
        return dict(kind="q", dim=dim, nc=size(7, 48) if dim == 2 else size(4, 16),
                    l=rng.choice([3, 4, 5]) if dim == 2 else rng.choice([2, 3]),
                    coef=rng.choice(["iid", "smooth"]), sigma=sigma,
                    load=rng.choice(["const", "cell"]),
                    reaction=rng.choice(["none", "const", "cell"]),
                    solver=rng.choice(["mfma", "mfma", "default"]),
                    want=rng.choice(["basis", "solution"]))
    if kind == "tensor":
        l = rng.choice([3, 4])
        return dict(kind="q", dim=3, nc=size(2, 8) if l == 3 else size(2, 4), l=l, coef="tensor",
                    sigma=round(rng.uniform(0.3, 0.9), 3), load=rng.choice(["const", "qp"]),
                    reaction="none", solver="cg", want="basis")
    if kind == "gradient":
        return dict(kind="q", dim=3, nc=size(4, 16), l=rng.choice([2, 3]),
                    coef=rng.choice(["iid", "smooth"]), sigma=sigma, load="const", reaction="none",
                    solver="mfma", want="gradient")
    if kind == "uneven":
        nc = size(6, 16)
        return dict(kind="uneven", dim=3, nc=nc, inclusions=max(4, nc ** 3 // rng.choice([10, 15])),
                    radius=round(rng.uniform(0.2, 0.4) / nc, 4), value=10.0 ** rng.choice([2, 3, 4]))
    if kind == "ned":
        return dict(kind="ned", nc=size(6, 32), l=rng.choice([2, 3, 4]), sigma=sigma)
    if kind == "rt":
        l = rng.choice([3, 4, 5])
        return dict(kind="rt", nc=size(6, 32) if l < 5 else size(6, 20), l=l,
                    coef=rng.choice(["scalar", "tensor"]), sigma=round(rng.uniform(0.3, 0.9), 3))
    alpha = round(rng.uniform(0.3, 0.9), 3)
    if kind == "rt3":
        l = rng.choice([2, 3, 4])
        return dict(kind="rt3", nc=size(2, {2: 12, 3: 6, 4: 4}[l]), l=l, alpha=alpha)
    l = rng.choice([2, 2, 3, 4])
    return dict(kind="nrt", nc=size(*{2: (3, 16), 3: (2, 3), 4: (1, 2)}[l]), l=l, alpha=alpha)


# --------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 2 + 1)


def _field(gen, dim, nc, N, sigma, corr):
    """Gaussian field (standard deviation sigma, correlation length corr of
    the domain, 0: iid) on the global fine grid, cut into per-cell blocks."""
    n = nc * N
    g = torch.randn((n,) * dim, generator=gen, device=DEV, dtype=F64)
    if corr > 0:
        k2 = sum(torch.meshgrid(*[torch.fft.fftfreq(n, device=DEV, dtype=F64) ** 2] * dim,
                                indexing="ij"))
        amp = torch.exp(-math.pi ** 2 * 2.0 * (corr * n) ** 2 * k2)
        g = torch.fft.ifftn(torch.fft.fftn(g) * torch.sqrt(amp)).real
        g = (g - g.mean()) / g.std()
    g = sigma * g
    if dim == 2:
        return g.reshape(nc, N, nc, N).permute(0, 2, 1, 3).reshape(nc * nc, N * N).contiguous()
    return g.reshape(nc, N, nc, N, nc, N).permute(0, 2, 4, 1, 3, 5).reshape(
        nc ** 3, N ** 3).contiguous()


def _points(dim, nc, l):
    """QGauss(2) points of every fine cell: (nc^dim, N^dim, 2^dim, dim)."""
    N = 1 << l
    i = torch.arange(nc ** dim, device=DEV)
    c = torch.arange(N ** dim, device=DEV)
    q = torch.arange(1 << dim, device=DEV)
    g = torch.tensor([0.5 - 0.5 / math.sqrt(3), 0.5 + 0.5 / math.sqrt(3)], device=DEV, dtype=F64)
    return torch.stack([((i // nc ** d % nc)[:, None, None] +
                         ((c // N ** d % N)[:, None] + g[q >> d & 1]) / N) / nc
                        for d in range(dim)], -1)


def _tensor(x, alpha, gen, inverse):
    """The oscillatory diagonal of the reference's Diffusion_A (frequencies
    17, 16, 15, a random phase per direction) turned by its Euler rotation (a
    rotation by pi/3 in 2-D), as the symmetric components per point."""
    dim = x.shape[-1]
    ph = torch.rand(dim, generator=gen, device=DEV, dtype=F64)
    fr = torch.tensor([17.0, 16.0, 15.0][:dim], device=DEV, dtype=F64)
    d = 1.0 - alpha * torch.sin(2 * math.pi * (fr * x + ph))
    if inverse:
        d = 1.0 / d
    if dim == 3:
        R = torch.as_tensor(F._euler_rotation(), device=DEV, dtype=F64)
        ij = ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))
    else:
        c, s = math.cos(math.pi / 3), math.sin(math.pi / 3)
        R = torch.tensor([[c, -s], [s, c]], device=DEV, dtype=F64)
        ij = ((0, 0), (0, 1), (1, 1))
    return torch.stack([(R[i] * R[j] * d).sum(-1) for i, j in ij], -1).contiguous()


def _levels(case, seed):
    """The levels of the mesh, made once around the cells that hold an
    inclusion, and centres in those cells from the seed."""
    nc = case["nc"]
    cell = np.floor(F.inclusion_centres(3, case["inclusions"], 0) * nc) / nc
    cen = cell + np.random.default_rng(seed).random(cell.shape) * (0.999 / nc)
    return cen, F.uneven_levels(3, nc, cell + 0.5 / nc, 1)


def _inputs(case, seed):
    """Device tensors of one case, by name."""
    gen, kind, nc = _gen(seed), case["kind"], case["nc"]
    if kind == "uneven":
        cen, lv = _levels(case, seed)
        blk = F.inclusion_blocks(3, nc, lv, cen, case["radius"], case["value"])
        return {"coef": torch.as_tensor(np.concatenate(blk), device=DEV), "levels": lv}
    l = case["l"]
    N = 1 << l
    if kind == "q":
        dim = case["dim"]
        n, nf = nc ** dim, N ** dim
        out = {}
        if case["coef"] == "tensor":
            x = _points(dim, nc, l)
            out["coef"] = _tensor(x, case["sigma"], gen, False)
        else:
            out["coef"] = torch.exp(_field(gen, dim, nc, N, case["sigma"],
                                           1 / 64 if case["coef"] == "smooth" else 0.0))
        if case["load"] == "cell":
            out["f"] = 1.0 + 0.5 * torch.randn(n, nf, generator=gen, device=DEV, dtype=F64)
        elif case["load"] == "qp":
            ph = torch.rand(dim, generator=gen, device=DEV, dtype=F64)
            out["f"] = torch.sin(2 * math.pi * (x + ph)).prod(-1).contiguous()
        if case["reaction"] == "cell":
            out["r"] = torch.rand(n, nf, generator=gen, device=DEV, dtype=F64) + 0.5
        if case["want"] == "gradient":
            t = torch.rand((nc + 1,) * dim, generator=gen, device=DEV, dtype=F64)
            out["target"] = (0.05 * t).reshape(-1).contiguous()
        return out
    if kind == "ned":
        n, nf = nc * nc, N * N
        return {"a": torch.exp(_field(gen, 2, nc, N, case["sigma"], 0.0)),
                "binv": torch.exp(_field(gen, 2, nc, N, 0.3, 0.0)),
                "r": torch.rand(n, nf, generator=gen, device=DEV, dtype=F64),
                "f": torch.randn(n, nf, 2, generator=gen, device=DEV, dtype=F64)}
    if kind == "rt":
        f = 1.0 + 0.5 * torch.randn(nc * nc, N * N, generator=gen, device=DEV, dtype=F64)
        if case["coef"] == "tensor":
            return {"a": _tensor(_points(2, nc, l), case["sigma"], gen, False), "f": f}
        return {"a": torch.exp(_field(gen, 2, nc, N, case["sigma"], 0.0)), "f": f}
    x = _points(3, nc, l)
    ainv = _tensor(x, case["alpha"], gen, True)
    ph = torch.rand(3, generator=gen, device=DEV, dtype=F64)
    if kind == "rt3":
        return {"ainv": ainv, "f": torch.sin(2 * math.pi * (x + ph)).prod(-1).contiguous()}
    y = x + 0.1 * ph
    b = 1.0 - case["alpha"] * torch.sin(2 * math.pi * (14 * x[..., 0] + ph[0]))
    p = y * (y - 1)
    f = 100.0 * torch.stack([(2 * y[..., 0] - 1) * p[..., 1] * p[..., 2],
                             (2 * y[..., 1] - 1) * p[..., 0] * p[..., 2],
                             (2 * y[..., 2] - 1) * p[..., 0] * p[..., 1]], -1)
    return {"ainv": ainv, "b": b.contiguous(), "f": f.contiguous()}


# --------------------------------------------------------------------------- passes
def _sizes(case):
    """(cells, bases, fine dofs per basis, fine cells per cell, dofs of a fine
    cell, entries of M per side) of a case with one level."""
    kind, nc = case["kind"], case["nc"]
    m = 1 << case["l"]
    if kind == "q":
        d = case["dim"]
        return nc ** d, 1 << d, (m + 1) ** d, m ** d, 1 << d, 1 << d
    if kind == "ned":
        return nc * nc, 8, (m + 1) ** 2 + 2 * m * (m + 1), m * m, 8, 8
    if kind == "rt":
        return nc * nc, 4, 2 * m * (m + 1), m * m, 4, 5
    nf = 3 * m * m * (m + 1)
    if kind == "rt3":
        return nc ** 3, 6, nf, m ** 3, 6, 7
    return nc ** 3, 18, nf + 3 * m * (m + 1) ** 2, m ** 3, 18, 18


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _empty(*shape):
    return torch.empty(shape, device=DEV, dtype=F64)


def prepare(case, seed):
    kind, nc = case["kind"], case["nc"]
    s = {"case": case, "in": _inputs(case, seed), "lib": L.load()}
    if kind == "uneven":
        h = UnevenBatch(F.coarse_vertices(3, nc), s["in"]["levels"])
        # the solver of every level is part of the plan that a program keeps
        h.set_coefficients(s["in"]["coef"])
        h.tune()
        n = nc ** 3
        s.update(h=h, out=[_empty(n, 8, 8), _empty(n, 8), _empty(int(h.basis_offsets[-1]))])
        return s
    l = case["l"]
    n, nb, nd, _, _, nm = _sizes(case)
    if kind == "q":
        dim = case["dim"]
        h = QBasisBatch(
            F.coarse_vertices(dim, nc), dim=dim, n_refine_local=l,
            coef_mode=L.COEF_TENSOR_QP if case["coef"] == "tensor" else L.COEF_SCALAR_CELL,
            rhs_mode={"const": L.RHS_CONST, "cell": L.RHS_CELL, "qp": L.RHS_QP}[case["load"]],
            reaction_mode={"none": L.REACTION_NONE, "const": L.REACTION_CONST,
                           "cell": L.REACTION_CELL}[case["reaction"]],
            reaction_const=1.0 if case["reaction"] == "const" else 0.0,
            solver=SOLVERS[case["solver"]])
        if "f" in s["in"]:
            h.set_rhs(s["in"]["f"])
        if "r" in s["in"]:
            h.set_reaction(s["in"]["r"])
        if case["want"] == "solution":
            out = [_empty((nc + 1) ** dim), _empty(n, nb), _empty(n, nd)]
        elif case["want"] == "gradient":
            out = [_empty(n, 1 << l * dim)]
            s["target"] = s["in"]["target"].cpu().numpy()
        else:
            out = [_empty(n, nb, nb), _empty(n, nb), _empty(n, nb, nd)]
        s.update(h=h, out=out)
        return s
    if kind == "ned":
        h = NedBasisBatch(F.coarse_vertices(2, nc), n_refine_local=l)
    elif kind == "rt":
        h = RTDQBasisBatch(F.coarse_vertices(2, nc), n_refine_local=l, coef_mode=(
            L.COEF_TENSOR_QP if case["coef"] == "tensor" else L.COEF_SCALAR_CELL))
    elif kind == "rt3":
        h = RTDQ3BasisBatch(F.coarse_vertices(3, nc), n_refine_local=l)
    else:
        h = NedRTBasisBatch(F.coarse_vertices(3, nc), n_refine_local=l)
    s.update(h=h, out=[_empty(n, nm, nm), _empty(n, nm), _empty(n, nb, nd)])
    return s


def run(s):
    case, h, lib, x, out = s["case"], s["h"], s["lib"], s["in"], s["out"]
    kind = case["kind"]
    if kind == "q":
        h.set_coefficient(x["coef"])
        h.run()
        if case["want"] == "solution":
            it, res = ctypes.c_int(0), ctypes.c_double(0.0)
            L.check(lib.msfec_coarse_solve(h._h, case["nc"], 1e-12, 1e-12, 100000, _ptr(out[0]),
                                           L.DEVICE, _ptr(out[1]), L.DEVICE, ctypes.byref(it),
                                           ctypes.byref(res)))
            h.set_global_weights(out[1], out=out[2])
        elif case["want"] == "gradient":
            J, g = h.adjoint_gradient(case["nc"], s["target"], out=out[0])
            return {"J": J, "gradient": g}
        else:
            L.check(lib.msfec_q_get_element(h._h, _ptr(out[0]), _ptr(out[1]), L.DEVICE))
            h.get_basis(out=out[2])
        return out
    if kind == "uneven":
        h.set_coefficients(x["coef"])
        element, basis = lib.msfec_qu_get_element, lib.msfec_qu_get_basis
    elif kind == "ned":
        h.set_coefficients(x["a"], x["binv"], x["r"], x["f"])
        element, basis = lib.msfec_ned_get_element, lib.msfec_ned_get_basis
    elif kind == "rt":
        h.set_coefficients(x["a"], x["f"])
        element, basis = lib.msfec_rt_get_element, lib.msfec_rt_get_basis
    elif kind == "rt3":
        L.check(lib.msfec_rt3_set_coefficients(h._h, _ptr(x["ainv"]), _ptr(x["f"]), L.DEVICE))
        element, basis = lib.msfec_rt3_get_element, lib.msfec_rt3_get_basis
    else:
        h.set_coefficients(x["ainv"], x["b"], None, x["f"])
        element, basis = lib.msfec_nrt_get_element, lib.msfec_nrt_get_basis
    h.run()
    L.check(element(h._h, _ptr(out[0]), _ptr(out[1]), L.DEVICE))
    L.check(basis(h._h, _ptr(out[2]), L.DEVICE))
    return out


def work(case):
    """Inputs read once and results written once.  The operations are one
    application of the fine operator to every basis (the residual that a
    solution has to make small) and one for the element matrix; what a solver
    adds to that is its own choice."""
    if case["kind"] == "uneven":
        n = case["nc"] ** 3
        fine = min(case["inclusions"], n)
        parts = [(fine, 4), ((n - fine) // 2, 2), ((n - fine) // 2, 3)]
    else:
        parts = [(_sizes(case)[0], case["l"])]
    by = fl = 0.0
    for cells, l in parts:
        c = dict(case, l=l)
        if case["kind"] == "uneven":
            c.update(kind="q", load="const", reaction="none", coef="iid", want="basis")
        n, nb, nd, nf, k, nm = _sizes(c)
        kind = c["kind"]
        if kind == "q":
            q = 1 << c["dim"]
            per = ((q * (3 if c["dim"] == 2 else 6) if c["coef"] == "tensor" else 1) +
                   {"const": 0, "cell": 1, "qp": q}[c["load"]] + (c["reaction"] == "cell"))
        else:
            per = {"ned": 5, "rt": 13 if c.get("coef") == "tensor" else 2, "rt3": 56, "nrt": 80}[kind]
        outs = nb * nd + nm * nm + nm
        if c.get("want") == "solution":
            outs = nd + nb + 1
        elif c.get("want") == "gradient":
            outs = nf
        by += 8.0 * cells * (per * nf + outs)
        fl += 4.0 * cells * nf * k * k * nb
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """All data and arithmetic are 64-bit.  Measured against the 64-bit
    reference below: direct solvers 1e-14 (element matrices 2e-14, Q_Ned 5e-11:
    the mass and curl blocks are 1e8 apart), the coarse CG and the iterative
    solvers 1e-13 to 2e-12 at their stopping rules, which bound the residual
    and not the error, so that another preconditioner ends elsewhere within
    them."""
    kind = case["kind"]
    if kind == "ned":
        return {"rel": 5e-10}
    if kind == "nrt":
        return {"rel": 1e-10}
    if kind == "uneven" or case.get("want") in ("solution", "gradient"):
        return {"rel": 2e-11}
    if kind == "rt3" or case.get("solver") == "cg":
        return {"rel": 1e-11}
    return {"rel": 1e-12}


# --------------------------------------------------------------------------- 64-bit reference
# Plain torch: fine-cell matrices Ke (cells, fine cells, k, k) by Gauss
# quadrature, a table T of each fine cell's dofs, and a solve of the interior
# rows: dense, conjugate gradients or MINRES, to rounding.
def _grid(dim, m):
    c = torch.arange(m ** dim, device=DEV)
    return [c // m ** d % m for d in range(dim)]


def _lex(i, n):
    """Lexicographic index of the coordinates i on a grid of n[d] points."""
    r = torch.zeros_like(i[0])
    for d in reversed(range(len(n))):
        r = r * n[d] + i[d]
    return r


def _gauss(dim):
    g = (0.5 - 0.5 / math.sqrt(3), 0.5 + 0.5 / math.sqrt(3))
    return [[g[q >> d & 1] for d in range(dim)] for q in range(1 << dim)]


def _hat(s, t):
    return t if s else 1.0 - t


def _nodes(dim, m):
    """Node table (fine cells, 2^dim)."""
    i = _grid(dim, m)
    return torch.stack([_lex([i[d] + (v >> d & 1) for d in range(dim)], [m + 1] * dim)
                        for v in range(1 << dim)], 1)


def _q1(dim, h):
    """Values and gradients of the Q1 shapes at the Gauss points: (q, v),
    (q, v, dim)."""
    val, gr = [], []
    for p in _gauss(dim):
        val.append([math.prod(_hat(v >> d & 1, p[d]) for d in range(dim)) for v in range(1 << dim)])
        gr.append([[math.prod((1.0 if v >> d & 1 else -1.0) / h if e == d else
                              _hat(v >> e & 1, p[e]) for e in range(dim)) for d in range(dim)]
                   for v in range(1 << dim)])
    return (torch.tensor(val, device=DEV, dtype=F64), torch.tensor(gr, device=DEV, dtype=F64))


def _full(t, dim):
    """Symmetric components (..., 3 or 6) -> matrices (..., dim, dim)."""
    idx = [[0, 1], [1, 2]] if dim == 2 else [[0, 1, 2], [1, 3, 4], [2, 4, 5]]
    return t[..., torch.tensor(idx, device=t.device)]


# deal.II's lines of the unit cube: axis and the fixed values of the two others
_LINES = [(1, 0, 0), (1, 1, 0), (0, 0, 0), (0, 1, 0), (1, 0, 1), (1, 1, 1), (0, 0, 1), (0, 1, 1),
          (2, 0, 0), (2, 1, 0), (2, 0, 1), (2, 1, 1)]


def _others(a):
    return [d for d in range(3) if d != a]


def _edge_table(m):
    """3-D edge table (fine cells, 12), and per edge its axis and position."""
    i = _grid(3, m)
    nx = m * (m + 1) ** 2
    cols = []
    for a, f1, f2 in _LINES:
        p = list(i)
        o = _others(a)
        p[o[0]], p[o[1]] = p[o[0]] + f1, p[o[1]] + f2
        cols.append(a * nx + _lex(p, [m if d == a else m + 1 for d in range(3)]))
    return torch.stack(cols, 1)


def _face_table(m):
    i = _grid(3, m)
    n1 = m * m * (m + 1)
    cols = []
    for a in range(3):
        for s in range(2):
            p = list(i)
            p[a] = p[a] + s
            cols.append(a * n1 + _lex(p, [m + 1 if d == a else m for d in range(3)]))
    return torch.stack(cols, 1)


def _edge_pos(m):
    """axis (ne,) and position (ne, 3) of every edge."""
    ax, pos = [], []
    for a in range(3):
        n = [m if d == a else m + 1 for d in range(3)]
        e = torch.arange(math.prod(n), device=DEV)
        ax.append(torch.full_like(e, a))
        pos.append(torch.stack([e % n[0], e // n[0] % n[1], e // (n[0] * n[1])], 1))
    return torch.cat(ax), torch.cat(pos)


def _face_pos(m):
    ax, pos = [], []
    for a in range(3):
        n = [m + 1 if d == a else m for d in range(3)]
        e = torch.arange(math.prod(n), device=DEV)
        ax.append(torch.full_like(e, a))
        pos.append(torch.stack([e % n[0], e // n[0] % n[1], e // (n[0] * n[1])], 1))
    return torch.cat(ax), torch.cat(pos)


def _ned_value(line, X, h):
    """(vector, curl) of the lowest-order Nedelec function of a line of a cube
    of side h at its reference point X."""
    a, f1, f2 = line
    o = _others(a)
    v1, v2 = _hat(f1, X[o[0]]), _hat(f2, X[o[1]])
    phi, gr, e = [0.0] * 3, [0.0] * 3, [0.0] * 3
    phi[a], e[a] = v1 * v2 / h, 1.0
    gr[o[0]] = (1.0 if f1 else -1.0) * v2 / h ** 2
    gr[o[1]] = v1 * (1.0 if f2 else -1.0) / h ** 2
    return phi, [gr[1] * e[2] - gr[2] * e[1], gr[2] * e[0] - gr[0] * e[2],
                 gr[0] * e[1] - gr[1] * e[0]]


def _rt_shapes(h):
    """Raviart-Thomas shapes at the Gauss points (q, 6, 3) and divergences (6)."""
    val = [[[_hat(f % 2, p[f // 2]) / h ** 2 if d == f // 2 else 0.0 for d in range(3)]
            for f in range(6)] for p in _gauss(3)]
    return (torch.tensor(val, device=DEV, dtype=F64),
            torch.tensor([(1.0 if f % 2 else -1.0) / h ** 3 for f in range(6)], device=DEV, dtype=F64))


def _apply(Ke, T, v):
    """The assembled operator on v (cells, r, dofs)."""
    out = torch.zeros_like(v)
    y = torch.matmul(v[:, :, T].transpose(1, 2), Ke.transpose(-1, -2).contiguous())
    out.index_add_(2, T.reshape(-1), y.transpose(1, 2).reshape(v.shape[0], v.shape[1], -1))
    return out


def _diag(Ke, T, nd):
    d = torch.zeros(Ke.shape[0], nd, device=Ke.device, dtype=F64)
    return d.index_add_(1, T.reshape(-1), torch.diagonal(Ke, dim1=-2, dim2=-1).reshape(Ke.shape[0], -1))


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _pcg(Ke, T, free, x, load=None, tol=1e-15):
    """Interior rows of K x = load for a (semi)definite K, x fixed elsewhere."""
    r = -_apply(Ke, T, x) * free
    if load is not None:
        r = r + load * free
    dinv = (free / _diag(Ke, T, x.shape[-1]).clamp_min(1e-300))[:, None]
    z = dinv * r
    p, rz = z.clone(), _dot(r, z)
    stop = tol ** 2 * rz
    for it in range(4000):
        if it % 16 == 0 and bool((rz <= stop).all()):
            break
        q = _apply(Ke, T, p) * free
        pq = _dot(p, q)
        al = torch.where(rz > stop, rz / torch.where(pq > 0, pq, torch.ones_like(pq)),
                         torch.zeros_like(rz))
        x = x + al * p
        r = r - al * q
        z = dinv * r
        new = _dot(r, z)
        p = z + torch.where(al != 0, new / rz.clamp_min(1e-300), torch.zeros_like(rz)) * p
        rz = torch.where(al != 0, new, rz)
    return x


def _minres(Ke, T, free, x, load, tol=1e-15):
    """Interior rows of a symmetric indefinite K x = load (Paige and Saunders),
    preconditioned by |diag K|."""
    dinv = (free / _diag(Ke, T, x.shape[-1]).abs().clamp_min(1e-300))[:, None]

    def safe(a, b):
        return torch.where(b.abs() > 0, a / torch.where(b.abs() > 0, b, torch.ones_like(b)),
                           torch.zeros_like(a))

    r2 = (load - _apply(Ke, T, x)) * free
    r1 = torch.zeros_like(r2)
    y = dinv * r2
    beta = _dot(r2, y).sqrt()
    beta0, old, dbar, eps = beta, torch.zeros_like(beta), torch.zeros_like(beta), torch.zeros_like(beta)
    phibar, cs, sn = beta, -torch.ones_like(beta), torch.zeros_like(beta)
    w1, w2 = torch.zeros_like(r2), torch.zeros_like(r2)
    for it in range(12000):
        if it % 32 == 0 and bool((phibar.abs() <= tol * beta0).all()):
            break
        v = safe(y, beta)
        y = _apply(Ke, T, v) * free
        if it > 0:
            y = y - safe(beta, old) * r1
        alfa = _dot(v, y)
        y = y - safe(alfa, beta) * r2
        r1, r2 = r2, y
        y = dinv * r2
        old, beta = beta, _dot(r2, y).clamp_min(0).sqrt()
        oeps, delta, gbar = eps, cs * dbar + sn * alfa, sn * dbar - cs * alfa
        eps, dbar = sn * beta, -cs * beta
        gam = torch.sqrt(gbar ** 2 + beta ** 2).clamp_min(1e-300)
        cs, sn = gbar / gam, beta / gam
        phi, phibar = cs * phibar, sn * phibar
        w = (v - oeps * w1 - delta * w2) / gam
        w1, w2 = w2, w
        x = x + phi * w
    return x


def _dense(Ke, T, free, x, load):
    """Interior rows by an equilibrated dense LU with one refinement step."""
    B, _, nd = x.shape
    A = torch.zeros(B, nd * nd, device=Ke.device, dtype=F64)
    A.index_add_(1, (T[:, :, None] * nd + T[:, None, :]).reshape(-1), Ke.reshape(B, -1))
    i = torch.nonzero(free).reshape(-1)
    A = A.reshape(B, nd, nd)[:, i][:, :, i]
    s = torch.diagonal(A, dim1=-2, dim2=-1).abs().rsqrt()
    # batches of small factorisations run on the host
    where = DEV if len(i) > 512 else "cpu"
    lu, piv = torch.linalg.lu_factor((s[:, :, None] * A * s[:, None, :]).contiguous().to(where))
    x = x.clone()
    for _ in range(3):
        r = (load - _apply(Ke, T, x))[:, :, i].transpose(1, 2)
        d = torch.linalg.lu_solve(lu, piv, (s[:, :, None] * r).contiguous().to(where))
        x[:, :, i] += (s[:, :, None] * d.to(DEV)).transpose(1, 2)
    return x


def _chunks(n, per_cell_bytes, limit=2e9):
    step = max(1, min(n, int(limit / per_cell_bytes)))
    return [slice(a, min(a + step, n)) for a in range(0, n, step)]


def _q_cells(dim, H, l, x, tensor, sl):
    """(Ke, F, T, free, G) of the cells sl: matrices, nodal loads, node table,
    interior mask and the coarse Q1 functions at the nodes."""
    m = 1 << l
    h = H / m
    val, gr = _q1(dim, h)
    w = h ** dim / (1 << dim)
    a = x["coef"][sl]
    if tensor:
        # one entry of the symmetric matrices at a time
        A = _full(a, dim)
        Ke = torch.stack([torch.stack([torch.einsum("cfqde,qde->cf", A, gr[:, i, :, None] *
                                                    gr[:, j, None, :]) for j in range(1 << dim)], -1)
                          for i in range(1 << dim)], -2) * w
    else:
        Ke = a[:, :, None, None] * torch.einsum("qid,qjd->ij", gr, gr) * w
    if "r" in x:
        Ke = Ke + x["r"][sl][:, :, None, None] * torch.einsum("qi,qj->ij", val, val) * w
    elif x.get("rconst"):
        Ke = Ke + x["rconst"] * torch.einsum("qi,qj->ij", val, val) * w
    T = _nodes(dim, m)
    nd = (m + 1) ** dim
    f = x.get("f")
    if f is None:
        Fe = torch.full((a.shape[0], m ** dim, 1 << dim), w, device=DEV, dtype=F64)
    elif f.dim() == 2:
        Fe = f[sl][:, :, None] * w * val.sum(0)
    else:
        Fe = torch.einsum("cfq,qi->cfi", f[sl], val) * w
    load = torch.zeros(a.shape[0], nd, device=DEV, dtype=F64).index_add_(
        1, T.reshape(-1), Fe.reshape(a.shape[0], -1))
    n = torch.arange(nd, device=DEV)
    p = [n // (m + 1) ** d % (m + 1) for d in range(dim)]
    free = torch.stack([(c > 0) & (c < m) for c in p]).all(0).to(F64)
    G = torch.stack([math.prod(((p[d].to(F64) / m) if v >> d & 1 else (1 - p[d].to(F64) / m))
                               for d in range(dim)) for v in range(1 << dim)])
    return Ke, load, T, free, G


def _q_exact(dim, H, l, x, tensor=False, adjoint=False):
    """M, b, Psi of every cell (and K_II^-1 F_I where the adjoint asks)."""
    n = x["coef"].shape[0]
    m, nb = 1 << l, 1 << dim
    Ms, bs, Ps, ws = [], [], [], []
    for sl in _chunks(n, 8 * m ** dim * nb * (4 * nb + (nb * 8 if tensor else 0))):
        Ke, load, T, free, G = _q_cells(dim, H, l, x, tensor, sl)
        psi = _pcg(Ke, T, free, G[None].repeat(Ke.shape[0], 1, 1))
        Ms.append(torch.matmul(psi, _apply(Ke, T, psi).transpose(1, 2).contiguous()))
        bs.append(torch.matmul(psi, load[:, :, None])[:, :, 0])
        Ps.append(psi)
        if adjoint:
            ws.append(_pcg(Ke, T, free, torch.zeros_like(load)[:, None], load[:, None])[:, 0])
    return torch.cat(Ms), torch.cat(bs), torch.cat(Ps), (torch.cat(ws) if adjoint else None)


def _coarse(dim, nc, M, rhs):
    """Assembled coarse system: the solve for nodal right-hand sides, zero on
    the boundary."""
    nn = (nc + 1) ** dim
    T = _nodes(dim, nc)
    K = torch.zeros(nn * nn, device=DEV, dtype=F64)
    K.index_add_(0, (T[:, :, None] * nn + T[:, None, :]).reshape(-1), M.reshape(-1))
    n = torch.arange(nn, device=DEV)
    free = torch.stack([(n // (nc + 1) ** d % (nc + 1) > 0) & (n // (nc + 1) ** d % (nc + 1) < nc)
                        for d in range(dim)]).all(0)
    i = torch.nonzero(free).reshape(-1)
    C = torch.linalg.cholesky(K.reshape(nn, nn)[i][:, i])

    def solve(r):
        u = torch.zeros(nn, device=DEV, dtype=F64)
        u[i] = torch.cholesky_solve(r[i][:, None], C)[:, 0]
        return u

    f = torch.zeros(nn, device=DEV, dtype=F64).index_add_(0, T.reshape(-1), rhs.reshape(-1))
    return T, free, f, solve


def _block_exact(parts, Ke, T, free, x, load, split, first, f, direct):
    """Bases of a mixed system whose rows from `split` on enter the symmetric
    form with the opposite sign, and the element matrix by blocks: bases below
    `first` enter through the dofs below `split`, the others through the rest."""
    if direct:
        x = _dense(Ke, T, free, x, load)
    else:
        sg = torch.ones(x.shape[-1], device=DEV, dtype=F64)
        sg[split:] = -1.0
        x = _minres(Ke * sg[T][None, :, :, None], T, free, x, load * sg)
    y = x.clone()
    y[:, :first, split:] = 0
    y[:, first:, :split] = 0
    M = torch.matmul(y, _apply(Ke, T, y).transpose(1, 2).contiguous())
    b = torch.matmul(y, f[:, :, None])[:, :, 0]
    b[:, :first] = 0
    parts.append((M, b, x))


def _join(parts):
    return [torch.cat([p[k] for p in parts]) for k in range(3)]


def _ned_exact(case, x):
    nc, m = case["nc"], 1 << case["l"]
    H = 1.0 / nc
    h = H / m
    i, j = _grid(2, m)
    ns, nh = (m + 1) ** 2, m * (m + 1)
    T = torch.cat([_nodes(2, m), torch.stack([ns + nh + j * (m + 1) + i, ns + nh + j * (m + 1) + i + 1,
                                              ns + j * m + i, ns + (j + 1) * m + i], 1)], 1)
    nd = ns + 2 * nh
    val, gr = _q1(2, h)
    ev = torch.tensor([[[0.0, (1 - p[0]) / h], [0.0, p[0] / h], [(1 - p[1]) / h, 0.0], [p[1] / h, 0.0]]
                       for p in _gauss(2)], device=DEV, dtype=F64)
    curl = torch.tensor([-1.0, 1.0, 1.0, -1.0], device=DEV, dtype=F64) / h ** 2
    w = h * h / 4
    mass = torch.einsum("qi,qj->ij", val, val) * w
    grad = torch.einsum("qid,qed->ie", gr, ev) * w          # (grad phi_i, v_e)
    cc = curl[:, None] * curl[None] * 4 * w
    em = torch.einsum("qed,qgd->eg", ev, ev) * w
    # boundary values of the 8 bases and the sources (v, grad phi_n)
    node = torch.arange(ns, device=DEV)
    X, Y = (node % (m + 1)).to(F64) / m, (node // (m + 1)).to(F64) / m
    phi = torch.stack([(X if v & 1 else 1 - X) * (Y if v >> 1 else 1 - Y) for v in range(4)])
    he, ve = torch.arange(nh, device=DEV), torch.arange(nh, device=DEV)
    hi, hj, vi, vj = he % m, he // m, ve % (m + 1), ve // (m + 1)
    G = torch.zeros(8, nd, device=DEV, dtype=F64)
    G[:4, :ns] = phi
    G[:4, ns:ns + nh] = phi[:, hj * (m + 1) + hi + 1] - phi[:, hj * (m + 1) + hi]
    G[:4, ns + nh:] = phi[:, (vj + 1) * (m + 1) + vi] - phi[:, vj * (m + 1) + vi]
    source = G.clone()
    source[:, :ns] = 0
    G[6, ns:ns + nh], G[7, ns:ns + nh] = (hj == 0) / m, (hj == m) / m
    G[4, ns + nh:], G[5, ns + nh:] = (vi == 0) / m, (vi == m) / m
    free = torch.cat([(X > 0) & (X < 1) & (Y > 0) & (Y < 1), (hj > 0) & (hj < m),
                      (vi > 0) & (vi < m)]).to(F64)
    mk = torch.zeros(1, m * m, 8, 8, device=DEV, dtype=F64)
    mk[..., 4:, 4:] = em
    load = _apply(mk, T, source[None])                      # edge mass times the gradient's edges
    parts = []
    for sl in _chunks(nc * nc, 24 * nd * nd):
        a, bi, r, f = x["a"][sl], x["binv"][sl], x["r"][sl], x["f"][sl]
        Ke = torch.zeros(a.shape[0], m * m, 8, 8, device=DEV, dtype=F64)
        Ke[..., :4, :4] = bi[..., None, None] * mass
        Ke[..., :4, 4:] = -grad
        Ke[..., 4:, :4] = grad.T
        Ke[..., 4:, 4:] = a[..., None, None] * cc + r[..., None, None] * em
        fe = torch.einsum("cfd,qed->cfe", f, ev) * w
        F_ = torch.zeros(a.shape[0], nd, device=DEV, dtype=F64).index_add_(
            1, T[:, 4:].reshape(-1), fe.reshape(a.shape[0], -1))
        _block_exact(parts, Ke, T, free, (G * (1 - free)).repeat(a.shape[0], 1, 1),
                     load.repeat(a.shape[0], 1, 1), ns, 4, F_, True)
    return _join(parts)


def _nrt_exact(case, x):
    nc, m = case["nc"], 1 << case["l"]
    H = 1.0 / nc
    h = H / m
    w = h ** 3 / 8
    ne = 3 * m * (m + 1) ** 2
    T = torch.cat([_edge_table(m), ne + _face_table(m)], 1)
    (ea, ep), (fa, fp) = _edge_pos(m), _face_pos(m)
    nd = ne + len(fa)
    ev = torch.tensor([[_ned_value(e, p, h)[0] for e in _LINES] for p in _gauss(3)], device=DEV, dtype=F64)
    ec = torch.tensor([[_ned_value(e, p, h)[1] for e in _LINES] for p in _gauss(3)], device=DEV, dtype=F64)
    fv, dv = _rt_shapes(h)
    cpl = torch.einsum("qfd,qed->fe", fv, ec) * w           # (v_f, curl tau_e)
    fm = torch.einsum("qfd,qgd->fg", fv, fv) * w
    # traces: line integrals of the coarse Nedelec, fluxes of the coarse
    # Raviart-Thomas functions; (v, curl N_n) = face mass times circulations
    G = torch.zeros(18, nd, device=DEV, dtype=F64)
    for n, (a, f1, f2) in enumerate(_LINES):
        o = _others(a)
        t = [ep[:, d].to(F64) / m for d in o]
        G[n, :ne] = (ea == a) * (t[0] if f1 else 1 - t[0]) * (t[1] if f2 else 1 - t[1]) / m
    coarse = G.clone()
    for f in range(6):
        G[12 + f, ne:] = ((fa == f // 2) & (fp.gather(1, fa[:, None])[:, 0] == (f % 2) * m)) / (m * m)
    efree = torch.stack([(ea == d) | ((ep[:, d] > 0) & (ep[:, d] < m)) for d in range(3)]).all(0)
    fpos = fp.gather(1, fa[:, None])[:, 0]
    free = torch.cat([efree, (fpos > 0) & (fpos < m)]).to(F64)
    kc = torch.zeros(1, m ** 3, 18, 18, device=DEV, dtype=F64)
    kc[..., 12:, :12] = cpl
    load = _apply(kc, T, coarse[None])
    parts = []
    for sl in _chunks(nc ** 3, 8 * m ** 3 * 18 * 18 * 6, 4e9):
        A, b, f = x["ainv"][sl], x["b"][sl], x["f"][sl]
        n = A.shape[0]
        Ke = torch.zeros(n, m ** 3, 18, 18, device=DEV, dtype=F64)
        Af = _full(A, 3)
        for e in range(12):
            t = torch.einsum("cfqde,qe->cfqd", Af, ev[:, e])
            Ke[..., :12, e] = torch.einsum("cfqd,qid->cfi", t, ev) * w
        Ke[..., 12:, :12] = cpl
        Ke[..., :12, 12:] = -cpl.T
        Ke[..., 12:, 12:] = b.sum(-1)[..., None, None] * (dv[:, None] * dv[None]) * w
        fe = torch.einsum("cfqd,qid->cfi", f, fv) * w
        F_ = torch.zeros(n, nd, device=DEV, dtype=F64).index_add_(
            1, T[:, 12:].reshape(-1), fe.reshape(n, -1))
        _block_exact(parts, Ke, T, free, (G * (1 - free)).repeat(n, 1, 1), load.repeat(n, 1, 1),
                     ne, 12, F_, False)
    return _join(parts)


def _flux_exact(nc, dim, l, MA, F_, curlT, C, TF, pfree, coarse):
    """Flux bases coarse + curl p, p minimising the A^-1 energy: MA the face
    masses (cells, fine cells, k, k), C (k, j) the circulation of a fine cell's
    potential dofs around its faces, curlT / TF the potential / face tables."""
    nb = 2 * dim
    nf = coarse.shape[-1]
    parts = []
    for sl in _chunks(nc ** dim, 8 * MA.shape[1] * nb * 3 * 24, 4e9):
        A = MA(sl) if callable(MA) else MA[sl]
        n = A.shape[0]
        Kp = torch.einsum("fi,...fg,gj->...ij", C, A, C)
        g = torch.einsum("cefg,bef->cbeg", A.transpose(-1, -2), coarse[:, TF])
        g = torch.einsum("cbeg,gj->cbej", g, C)
        load = torch.zeros(n, nb, pfree.shape[0], device=DEV, dtype=F64).index_add_(
            2, curlT.reshape(-1), -g.reshape(n, nb, -1))
        p = _pcg(Kp, curlT, pfree, torch.zeros_like(load), load)
        # every face takes its circulation from one fine cell that holds it
        flat = TF.reshape(-1)
        owner = torch.zeros(nf, dtype=torch.long, device=DEV).scatter_(
            0, flat, torch.arange(flat.numel(), device=DEV))
        s = coarse[None] + torch.einsum("cbej,fj->cbef", p[:, :, curlT], C).reshape(n, nb, -1)[:, :, owner]
        M = torch.zeros(n, nb + 1, nb + 1, device=DEV, dtype=F64)
        M[:, :nb, :nb] = torch.matmul(s, _apply(A, TF, s).transpose(1, 2).contiguous())
        div = (s[:, :, TF] * torch.tensor([-1.0, 1.0] * dim, device=DEV, dtype=F64)).sum((-1, -2))
        M[:, nb, :nb], M[:, :nb, nb] = div, -div
        b = torch.zeros(n, nb + 1, device=DEV, dtype=F64)
        b[:, nb] = F_[sl]
        parts.append((M, b, s))
    return _join(parts)


def _rt_exact(case, x):
    nc, m = case["nc"], 1 << case["l"]
    h = 1.0 / nc / m
    i, j = _grid(2, m)
    nv = m * (m + 1)
    TF = torch.stack([j * (m + 1) + i, j * (m + 1) + i + 1, nv + j * m + i, nv + (j + 1) * m + i], 1)
    # flux of curl psi = (d_y psi, -d_x psi) through the faces from the nodes
    C = torch.tensor([[-1., 0, 1, 0], [0, -1, 0, 1], [1, -1, 0, 0], [0, 0, 1, -1]], device=DEV, dtype=F64)
    fv = torch.tensor([[[(1 - p[0]) / h, 0], [p[0] / h, 0], [0, (1 - p[1]) / h], [0, p[1] / h]]
                       for p in _gauss(2)], device=DEV, dtype=F64)
    w = h * h / 4
    a = x["a"]
    if case["coef"] == "tensor":
        Ai = torch.linalg.inv(_full(a, 2))
    else:
        Ai = (1 / a)[:, :, None, None, None] * torch.eye(2, device=DEV, dtype=F64).repeat(4, 1, 1)
    MA = torch.einsum("qid,cfqde,qje->cfij", fv, Ai, fv) * w
    e = torch.arange(nv, device=DEV)
    P, Q = (e % (m + 1)).to(F64) / m, (e // m).to(F64) / m
    coarse = torch.zeros(4, 2 * nv, device=DEV, dtype=F64)
    coarse[0, :nv], coarse[1, :nv], coarse[2, nv:], coarse[3, nv:] = (
        (1 - P) / m, P / m, (1 - Q) / m, Q / m)
    n = torch.arange((m + 1) ** 2, device=DEV)
    I, J = n % (m + 1), n // (m + 1)
    pfree = ((I > 0) & (I < m) & (J > 0) & (J < m)).to(F64)
    return _flux_exact(nc, 2, case["l"], MA, x["f"].sum(1) * h * h, _nodes(2, m), C, TF, pfree, coarse)


def _rt3_exact(case, x):
    nc, m = case["nc"], 1 << case["l"]
    h = 1.0 / nc / m
    w = h ** 3 / 8
    fv, _ = _rt_shapes(h)
    Af = _full(x["ainv"], 3)
    MA = torch.stack([torch.einsum("cfqd,qid->cfi", torch.einsum("cfqde,qe->cfqd", Af, fv[:, g]), fv)
                      for g in range(6)], -1) * w
    # the flux of curl p through a face: its four edges with the right-hand rule
    C = torch.zeros(6, 12, device=DEV, dtype=F64)
    for e, line in enumerate(_LINES):
        o = _others(line[0])
        for f in range(6):
            a, s = f // 2, f % 2
            if a in o and line[1 + o.index(a)] == s:
                other = [d for d in o if d != a][0]
                side = line[1 + o.index(other)]
                # flux of the constant-tangent edge function: +-1 from curl = grad x e
                sign = 1.0 if (other, line[0], a) in ((0, 1, 2), (1, 2, 0), (2, 0, 1)) else -1.0
                C[f, e] = sign * (1.0 if side else -1.0)
    fa, fp = _face_pos(m)
    t = fp.gather(1, fa[:, None])[:, 0].to(F64) / m
    coarse = torch.stack([(fa == f // 2) * (t if f % 2 else 1 - t) / (m * m) for f in range(6)])
    ea, ep = _edge_pos(m)
    pfree = torch.stack([(ea == d) | ((ep[:, d] > 0) & (ep[:, d] < m)) for d in range(3)]).all(0).to(F64)
    return _flux_exact(nc, 3, case["l"], MA, x["f"].sum((1, 2)) * w, _edge_table(m), C,
                       _face_table(m), pfree, coarse)


def exact(case, seed):
    x, kind, nc = _inputs(case, seed), case["kind"], case["nc"]
    if kind == "ned":
        return _ned_exact(case, x)
    if kind == "rt":
        return _rt_exact(case, x)
    if kind == "rt3":
        return _rt3_exact(case, x)
    if kind == "nrt":
        return _nrt_exact(case, x)
    if kind == "uneven":
        lv = torch.as_tensor(x["levels"], device=DEV, dtype=torch.long)
        co = torch.cumsum(torch.cat([torch.zeros_like(lv[:1]), 8 ** lv]), 0)
        po = torch.cumsum(torch.cat([torch.zeros_like(lv[:1]), 8 * (2 ** lv + 1) ** 3]), 0)
        M, b = _empty(nc ** 3, 8, 8), _empty(nc ** 3, 8)
        P = _empty(int(po[-1]))
        for l in sorted(set(x["levels"].tolist())):
            cells = torch.nonzero(lv == l).reshape(-1)
            a = x["coef"][co[cells][:, None] + torch.arange(8 ** l, device=DEV)]
            M[cells], b[cells], psi, _ = _q_exact(3, 1.0 / nc, l, {"coef": a})
            P[po[cells][:, None] + torch.arange(8 * ((1 << l) + 1) ** 3, device=DEV)] = psi.flatten(1)
        return [M, b, P]
    dim, l = case["dim"], case["l"]
    if case["reaction"] == "const":
        x["rconst"] = 1.0
    grad = case["want"] == "gradient"
    M, b, P, W = _q_exact(dim, 1.0 / nc, l, x, case["coef"] == "tensor", grad)
    if case["want"] == "basis":
        return [M, b, P]
    T, free, f, solve = _coarse(dim, nc, M, b)
    u = solve(f)
    if not grad:
        return [u, u[T], torch.matmul(u[T][:, None], P)[:, 0]]
    r = torch.where(free, u - x["target"], torch.zeros_like(u))
    v = solve(r)
    ut = torch.matmul(u[T][:, None], P)[:, 0] + W
    vt = torch.matmul(v[T][:, None], P)[:, 0]
    m = 1 << l
    _, gr = _q1(dim, 1.0 / nc / m)
    K = torch.einsum("qid,qjd->ij", gr, gr) * (1.0 / nc / m) ** dim / (1 << dim)
    N = _nodes(dim, m)
    g = -x["coef"] * ((vt[:, N] @ K) * ut[:, N]).sum(-1)
    return {"J": 0.5 * float((r * r).sum()), "gradient": g}
