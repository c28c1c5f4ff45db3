"""The sparse singular part reads no regular-rule points: on a new grid of 81920 cells it builds and
uploads the cells' records (21 MB), numbers and adjacent pairs (18 MB), and not the 37 points of every
cell (97 MB and more). Its values do not depend on the regular rule."""
import numpy as np
import pytest
import torch

from bempp_amd.assembly.boundary import BoundaryAssemblerOptions, OperatorType, create_laplace_assembler
from bempp_amd.element import Continuity, Family, ReferenceCellType, create_family
from bempp_amd.function_space import function_space
from bempp_amd.shapes import icosphere

pytestmark = pytest.mark.gpu


def _singular(level, nq):
    o = BoundaryAssemblerOptions()
    o.set_regular_quadrature_degree(ReferenceCellType.Triangle, nq)
    s = function_space(icosphere(level), create_family(Family.Lagrange, 0, Continuity.Discontinuous))
    return s, create_laplace_assembler(OperatorType.SingleLayer, o).assemble_singular(s, s)


def test_memory():
    _singular(1, 37)  # tables and code that every grid shares
    before = torch.cuda.mem_get_info()[0]
    s, m = _singular(6, 37)
    assert m.shape == (81920, 81920)
    assert before - torch.cuda.mem_get_info()[0] <= 72e6


def test_values():
    assert np.array_equal(_singular(2, 6)[1].toarray(), _singular(2, 37)[1].toarray())
