"""Two cells that cross at their common centroid, in every phase tier: the entries between them against the
oracle, 1e-12 relative as for every FP64 operator (rules without a point at the centroid)."""
import numpy as np
import pytest

import oracle_lib as O
from bempp_amd.assembly.boundary import (BoundaryAssemblerOptions, OperatorType, Precision, create_helmholtz_assembler)
from bempp_amd.element import Continuity, Family, ReferenceCellType, create_family
from bempp_amd.function_space import function_space
from bempp_amd.grid import Grid

pytestmark = pytest.mark.gpu

OPS = {"single_layer": OperatorType.SingleLayer, "double_layer": OperatorType.DoubleLayer,
       "adjoint_double_layer": OperatorType.AdjointDoubleLayer, "hypersingular": OperatorType.Hypersingular}
POINTS = np.array([[0.0, 0, 0], [3, 0, 0], [0, 3, 0], [2, 1, 1], [0, 1, 1], [1, 1, -2]])  # both centroids (1, 1, 0)
CELLS = np.array([[0, 1, 2], [3, 4, 5]])


@pytest.mark.parametrize("k", [0.05, 0.12, 0.3, -0.3, 3.0])
@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("degree", [0, 1])
@pytest.mark.parametrize("nq", [3, 6])
@pytest.mark.parametrize("precision", [Precision.FP64, Precision.Mixed])
def test_crossing(k, op, degree, nq, precision):
    o = BoundaryAssemblerOptions()
    o.set_regular_quadrature_degree(ReferenceCellType.Triangle, nq)
    o.set_precision(precision)
    a = create_helmholtz_assembler(k, OPS[op], o)
    s = function_space(Grid(POINTS, CELLS), create_family(Family.Lagrange, degree, Continuity.Standard if degree else
                                                          Continuity.Discontinuous))
    n = 3 if degree else 1
    R = O.assemble("helmholtz", op, POINTS, CELLS, test=(degree, degree == 1), trial=(degree, degree == 1), k=k, nq=nq,
                   nsing=4)[:n, n:]
    assert np.linalg.norm(a.assemble(s, s)[:n, n:] - R) <= 1e-12 * np.linalg.norm(R)
    if degree == 0:
        assert abs(a.apply(s, s, np.array([0.0, 1.0], dtype=complex))[0] - R[0, 0]) <= 1e-12 * abs(R[0, 0])


@pytest.mark.parametrize("k", [0.05, 0.12, 0.3])
def test_gradient(k):
    o = BoundaryAssemblerOptions()
    o.set_regular_quadrature_degree(ReferenceCellType.Triangle, 3)
    a = create_helmholtz_assembler(k, OperatorType.SingleLayer, o)
    s = function_space(Grid(POINTS, CELLS), create_family(Family.Lagrange, 0, Continuity.Discontinuous))
    assert np.isfinite(a.shape_gradient(s, s, np.array([1.0, 2j]), np.array([1j, 1.0]))).all()
