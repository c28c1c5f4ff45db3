"""Mixed precision on P1 spaces whose 64-cell blocks have many DOFs (a torus numbered in rows: 66 a
block): these stay in FP64, so the entries are those of Precision.FP64, 1e-12 relative (order of the
additions)."""
import pytest
import torch

from bempp_amd.assembly.boundary import (BoundaryAssemblerOptions, OperatorType, Precision, create_helmholtz_assembler,
                                         create_laplace_assembler)
from bempp_amd.element import Continuity, Family, ReferenceCellType, create_family
from bempp_amd.function_space import function_space
from bempp_amd.grid import Grid
from test_gpu_tile_parts import _torus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [None, 2.0])
@pytest.mark.parametrize("op", [OperatorType.SingleLayer, OperatorType.DoubleLayer, OperatorType.Hypersingular])
@pytest.mark.parametrize("test_degree", [0, 1])
def test_row_numbering(k, op, test_degree):
    p, c = _torus(40, 40)
    g = Grid(p, c)
    test, trial = (function_space(g, create_family(Family.Lagrange, d,
                                                   Continuity.Standard if d else Continuity.Discontinuous))
                   for d in (test_degree, 1))
    M = []
    for precision in (Precision.Mixed, Precision.FP64):
        o = BoundaryAssemblerOptions()
        o.set_regular_quadrature_degree(ReferenceCellType.Triangle, 6)
        o.set_precision(precision)
        a = create_laplace_assembler(op, o) if k is None else create_helmholtz_assembler(k, op, o)
        M.append(a.assemble_device(trial, test))
    assert torch.linalg.norm(M[0] - M[1]) <= 1e-12 * torch.linalg.norm(M[1])
