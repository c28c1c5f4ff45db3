"""Matrix-free products with an infinite entry: every entry of a single-layer matrix is positive, so every
entry of the product is infinite (none NaN), at adjacent cells too, which two kernels share."""
import numpy as np
import pytest

from bempp_amd.assembly.boundary import (BoundaryAssemblerOptions, OperatorType, create_laplace_assembler)
from bempp_amd.element import Continuity, Family, ReferenceCellType, create_family
from bempp_amd.function_space import function_space
from bempp_amd.grid import Grid
from test_gpu_tile_parts import _torus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu,nv", [(5, 5), (13, 5), (31, 7)])
@pytest.mark.parametrize("nq", [6, 16])
@pytest.mark.parametrize("at", [0, -1])
@pytest.mark.parametrize("transpose", [False, True])
def test_infinite_entry(nu, nv, nq, at, transpose):
    o = BoundaryAssemblerOptions()
    o.set_regular_quadrature_degree(ReferenceCellType.Triangle, nq)
    a = create_laplace_assembler(OperatorType.SingleLayer, o)
    g = Grid(*_torus(nu, nv))
    s = function_space(g, create_family(Family.Lagrange, 0, Continuity.Discontinuous))
    u = np.ones(len(g.cells))
    u[at] = np.inf
    assert np.isposinf(a.apply(s, s, u, transpose=transpose)).all()
