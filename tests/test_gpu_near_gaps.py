"""Cells that do not touch but are much nearer to each other than their size: two parallel sheets a
fraction of a cell apart, as one grid and as two. The entries between the sheets against the
oracle, which takes distances from differences of coordinates: 1e-12 relative, as for every
operator in FP64 (sums of at most 37^2 smooth terms)."""
import numpy as np
import pytest

import oracle_lib as O
from bempp_amd.assembly.boundary import (BoundaryAssemblerOptions, OperatorType, create_helmholtz_assembler,
                                         create_laplace_assembler)
from bempp_amd.element import Continuity, Family, ReferenceCellType, create_family
from bempp_amd.function_space import function_space
from bempp_amd.grid import Grid

pytestmark = pytest.mark.gpu

OPS = {"single_layer": OperatorType.SingleLayer, "double_layer": OperatorType.DoubleLayer,
       "adjoint_double_layer": OperatorType.AdjointDoubleLayer, "hypersingular": OperatorType.Hypersingular}


def _sheet(n, m, z, size=4):
    """n x m squares of side 1/4 in the plane z, as triangles or quadrilaterals."""
    x, y = np.meshgrid(np.arange(n + 1) * 0.25, np.arange(m + 1) * 0.25, indexing="ij")
    p = np.stack([x, y, np.full_like(x, z)], -1).reshape(-1, 3)
    i, j = np.meshgrid(np.arange(n), np.arange(m), indexing="ij")
    a = (i * (m + 1) + j).ravel()
    b, c, d = a + m + 1, a + 1, a + m + 2
    if size == 4:
        return p, np.stack([a, b, c, d], -1)
    return p, np.stack([np.stack([a, b, d], -1), np.stack([a, d, c], -1)], 1).reshape(-1, 3)


def _two(gap, size):
    (p, c), (q, _) = _sheet(5, 4, 0.0, size), _sheet(5, 4, gap, size)
    return p, c, np.concatenate([p, q]), np.concatenate([c, c + len(p)])


def _assembler(op, k, nq, cell):
    o = BoundaryAssemblerOptions()
    o.set_regular_quadrature_degree(cell, nq)
    return create_laplace_assembler(OPS[op], o) if k is None else create_helmholtz_assembler(k, OPS[op], o)


def _space(g, degree, continuous):
    return function_space(g, create_family(Family.Lagrange, degree,
                                           Continuity.Standard if continuous else Continuity.Discontinuous))


GAPS = [0.25 * 1e-1, 0.25 * 1e-3, 0.25 * 1e-5]


@pytest.mark.parametrize("gap", GAPS)
@pytest.mark.parametrize("k", [None, 1.0, 2.5, -6.0, 40.0])  # phase tiers 2 (or 1), 1, 3, 0 by the rule
@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("degree,continuous,nq", [(1, True, 1), (1, True, 3), (1, True, 6), (1, True, 7), (1, True, 16),
                                                  (1, False, 3), (0, False, 16), (0, False, 37)])
def test_dense(gap, k, op, degree, continuous, nq):
    if op == "hypersingular" and degree == 0:
        pytest.skip("the same sums as the single layer")
    p, c, pts, cells = _two(gap, 3)
    kind = "laplace" if k is None else "helmholtz"
    sp = (degree, continuous)
    R = O.assemble(kind, op, pts, cells, test=sp, trial=sp, k=k or 0.0, nq=nq, nsing=2)
    n = R.shape[0] // 2
    R = R[:n, n:]
    a = _assembler(op, k, nq, ReferenceCellType.Triangle)
    one = _space(Grid(pts, cells), *sp)
    A = a.assemble(one, one)[:n, n:]
    low, high = _space(Grid(p, c), *sp), _space(Grid(p + [0.0, 0.0, gap], c), *sp)
    for x in (A, a.assemble(high, low)):
        assert np.linalg.norm(x - R) <= 1e-12 * np.linalg.norm(R)


@pytest.mark.parametrize("gap", GAPS)
@pytest.mark.parametrize("k", [None, 1.0, 2.5, -6.0, 40.0])
@pytest.mark.parametrize("op", ["single_layer", "double_layer", "adjoint_double_layer"])
@pytest.mark.parametrize("nq", [1, 3, 6, 7, 16])
def test_apply(gap, k, op, nq):
    p, c, pts, cells = _two(gap, 3)
    R = O.assemble("laplace" if k is None else "helmholtz", op, pts, cells, k=k or 0.0, nq=nq, nsing=2)
    n = len(c)
    u = np.random.default_rng(nq).uniform(0.5, 1.5, n).astype(R.dtype)
    ref = R[:n, n:] @ u
    a = _assembler(op, k, nq, ReferenceCellType.Triangle)
    low, high = _space(Grid(p, c), 0, False), _space(Grid(p + [0.0, 0.0, gap], c), 0, False)
    one = _space(Grid(pts, cells), 0, False)
    for y in (a.apply(high, low, u), a.apply(one, one, np.concatenate([0 * u, u]))[:n]):
        assert np.linalg.norm(y - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("gap", GAPS)
@pytest.mark.parametrize("k", [None, 0.5, 1.0, -3.0, 20.0])
@pytest.mark.parametrize("nq", [4, 16])
def test_quadrilaterals(gap, k, nq):
    p, c, pts, cells = _two(gap, 4)
    R = O.assemble_cells("laplace" if k is None else "helmholtz", "single_layer", pts, cells, k=k or 0.0, nq_quad=nq,
                         part="regular")
    n = len(c)
    R = R[:n, n:]
    a = _assembler("single_layer", k, nq, ReferenceCellType.Quadrilateral)
    one = _space(Grid(pts, cells), 0, False)
    low, high = _space(Grid(p, c), 0, False), _space(Grid(p + [0.0, 0.0, gap], c), 0, False)
    for x in (a.assemble(one, one)[:n, n:], a.assemble(high, low)):
        assert np.linalg.norm(x - R) <= 1e-12 * np.linalg.norm(R)
