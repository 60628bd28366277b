"""The pair-lattice kernel on device 0 at the sizes where its tiles can go wrong:
meshes of one cell, one row more or less than a tile in a direction, part
boundaries inside a tile, no Dirichlet boundary, and each form of the
coefficient (constant, per cell, at the quadrature points) and source; against
the oracle.  Values are sums of at most 8 x 27 products of 64-bit numbers:
1e-12 of the largest entry."""
import numpy as np
import pytest

import oracle
from _helpers import STRUCT_KEYS, rel_err
from gridap_amd import AssemblyBatch, problem_from_workload
from gridap_amd import workloads as W

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(11)


def case(cells, parts, order, coef, dirichlet=True, strategy="sub", qdeg=None):
    dim = len(cells)
    p = dict(dim=dim, order=order, qdeg=qdeg or 2 * order, cells=cells, parts=parts, domain=(0.0, 1.3, -0.2, 0.7, 0.1, 2.0)[:2 * dim],
             strategy=strategy, coef_const=1.7, modes=np.zeros((0, 5)), rhs="const", rhs_const=0.9, dirichlet=dirichlet,
             uD=(0.3, 1.1, -0.6, 0.8 if dim == 3 else 0.0))
    if coef in ("points", "manufactured"):
        p["modes"] = W.fourier_modes(5, 5, 3, 0.4)
        if dim == 2:
            p["modes"][:, 2] = 0.0
        p["rhs"] = "manufactured" if coef == "manufactured" else "const"
    if coef == "cells":
        p["cell_kappa"] = np.exp(RNG.normal(size=int(np.prod(cells))))
    if coef == "const-manufactured":
        p["rhs"] = "manufactured"  # f = 0
    return p


CASES = [
    # Q2 tiles are 4 x 4 x 2 cells in 3D and 8 x 8 in 2D, Q1 tiles 15 x 7 x 3 (4 for kappa per cell) and 16 x 16 rows
    case((4, 4, 2), (1, 1, 1), 2, "manufactured"), case((5, 3, 3), (2, 1, 1), 2, "manufactured"),
    case((9, 8, 4), (2, 2, 1), 2, "cells"), case((1, 1, 1), (1, 1, 1), 2, "points", dirichlet=False),
    # thin: every row shorter than one 64-entry chunk; and rows of both chunks in front of ghost rows, which stay zero
    case((1, 1, 5), (1, 1, 2), 2, "cells", dirichlet=False), case((6, 3, 3), (2, 1, 1), 2, "points", dirichlet=False),
    case((2, 1, 5), (1, 1, 2), 2, "const", dirichlet=False), case((4, 5, 3), (1, 1, 1), 2, "points", strategy="full", qdeg=2),
    case((8, 4, 2), (1, 2, 1), 2, "const-manufactured", dirichlet=False),
    case((16, 8, 4), (1, 1, 1), 1, "manufactured"), case((17, 9, 5), (2, 1, 2), 1, "cells"),
    case((15, 7, 3), (1, 1, 1), 1, "points", dirichlet=False), case((31, 2, 7), (3, 1, 1), 1, "const"),
    case((1, 2, 1), (1, 1, 1), 1, "const", dirichlet=False), case((2, 2, 2), (2, 1, 1), 1, "cells", strategy="full"),
    case((8, 8), (1, 1), 2, "manufactured"), case((9, 17), (2, 1), 2, "cells"), case((1, 1), (1, 1), 2, "points", dirichlet=False),
    case((16, 7), (1, 2), 2, "points", qdeg=2), case((17, 16), (1, 1), 1, "manufactured"),
    case((18, 33), (2, 2), 1, "cells", strategy="full"), case((15, 2), (1, 1), 1, "const", dirichlet=False),
    case((16, 16), (1, 1), 1, "points", qdeg=4),
]


def ident(p):
    return f"{p['dim']}d-q{p['order']}-{'x'.join(map(str, p['cells']))}-{'x'.join(map(str, p['parts']))}-{p['strategy']}" \
           f"-{'cells' if 'cell_kappa' in p else ('modes' if len(p['modes']) else 'const')}-{p['rhs']}"


def assembled_matches_oracle(gpu_ctx, p, tol=1e-12):
    print("lattice kernel", ident(p), flush=True)
    q = dict(p)
    kappa = q.pop("cell_kappa", None)
    r = oracle.run(dict(q, cell_kappa=kappa) if kappa is not None else q)
    assem, data = problem_from_workload(gpu_ctx, q)
    prob = assem._problem_for(data)
    if kappa is not None:
        prob.set_cell_coefficient(kappa)
    for _ in range(2):  # a second pass over the same buffers
        prob.numeric()
    prob.sync()
    for k, P in enumerate(r.parts):
        Q = prob.export_part(k)
        for key in STRUCT_KEYS:
            assert np.array_equal(P[key], Q[key]), (k, key)
        if len(P["val"]):
            assert rel_err(Q["val"], P["val"]) <= tol
        assert np.all(Q["val"][Q["rowptr"][P["n_own"]]:] == 0.0)
        if len(P["b"]):
            assert np.abs(Q["b"] - P["b"]).max() <= tol * max(np.abs(P["b"]).max(), np.abs(P["val"]).max())
    prob.close()


@pytest.mark.parametrize("p", CASES, ids=ident)
def test_lattice_kernel_matches_oracle(gpu_ctx, p):
    assembled_matches_oracle(gpu_ctx, p)


# more lines in y, in z than a grid holds blocks: one beyond the limit and the padding of the last tile
@pytest.mark.parametrize("p", [case((3, 65600), (1, 2), 1, "cells"), case((2, 33000), (2, 1), 2, "const"),
                               case((2, 65537, 2), (1, 2, 1), 1, "const"), case((2, 2, 65537), (1, 1, 2), 1, "cells")],
                         ids=ident)
def test_long_boxes_match_oracle(gpu_ctx, p):
    # the oracle takes cell geometry from coordinates: a cell's width as a difference of coordinates n times as large
    # is off by up to n 2^-52 of itself (2D Q1 3 x 65000, cells of unit width: the oracle's b is 3.6e-12 of its
    # largest entry from the closed form in extended precision, the kernel's 7e-16)
    assembled_matches_oracle(gpu_ctx, p, tol=1e-12 + max(p["cells"]) * p["order"] * 2.0**-52)


def check(r, prob):
    for k, P in enumerate(r.parts):
        Q = prob.export_part(k)
        if len(P["val"]):
            assert rel_err(Q["val"], P["val"]) <= 1e-12, k
        if len(P["b"]):
            assert np.abs(Q["b"] - P["b"]).max() <= 1e-12 * max(np.abs(P["b"]).max(), np.abs(P["val"]).max()), k


# chunks of 8 (up to 8 modes) and of 16, whole and ragged, with and without the source's sum; lines of 64 points and more
@pytest.mark.parametrize("nmodes", [1, 8, 9, 16, 17])
@pytest.mark.parametrize("rhs", ["const", "manufactured"])
def test_coefficient_mode_chunks_match_oracle(gpu_ctx, nmodes, rhs):
    p = dict(case((33, 4, 3), (2, 1, 1), 1, "points"), rhs=rhs)
    p["modes"] = W.fourier_modes(nmodes, nmodes, 3, 0.4)
    r = oracle.run(p)
    assem, data = problem_from_workload(gpu_ctx, p)
    prob = assem._problem_for(data)
    # and the other kernels, which read f at the points also where it is constant
    for variant in (2, 1, 2, 0):
        prob.set_kernel(variant)
        prob.numeric()
        prob.sync()
        check(r, prob)
    prob.close()


@pytest.mark.parametrize("few", [True, False], ids=["up to 8 modes", "more"])
@pytest.mark.parametrize("source", [False, True], ids=["f constant", "f varies"])
def test_mixed_batch_matches_oracle(gpu_ctx, few, source):
    """Every tile shape and form of the coefficient in one batch, with a problem
    that no pair lattice takes beside them."""
    ps = [case((6, 5, 4), (2, 1, 1), 1, "points"), case((5, 4, 3), (1, 2, 1), 2, "points"),
          case((17, 9), (2, 1), 1, "points"), case((9, 8), (1, 1), 2, "points"), case((16, 8, 4), (1, 1, 1), 1, "const"),
          case((4, 3, 3), (1, 1, 1), 2, "const"), case((7, 7, 5), (1, 1, 2), 1, "const")]
    if not few:
        ps[0]["modes"] = W.fourier_modes(12, 12, 3, 0.4)
    if source:
        ps[1]["rhs"] = "manufactured"
        ps[2]["rhs"] = "manufactured"
    refs, probs = [oracle.run(p) for p in ps], []
    b = AssemblyBatch(gpu_ctx)
    for k, p in enumerate(ps):
        assem, data = problem_from_workload(gpu_ctx, p)
        probs.append(assem._problem_for(data))
        b.add(probs[-1])
    b.autotune(1)
    probs[-1].set_kernel(1)
    b.capture()
    for _ in range(3):
        b.launch()
        b.sync()
        for r, prob in zip(refs, probs):
            check(r, prob)
    b.close()
    for prob in probs:
        prob.close()
