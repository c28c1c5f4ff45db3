"""The sparse singular part reads no regular-rule points: on a new grid of 81920 cells it takes as much
device memory with the 37-point rule as with the 1-point one, where the cells' points of the former are
97 MB and of the latter 2.6 MB. 16 MB of slack: the allocator's granularity of 2 MiB, in no more than
eight allocations. Its values do not depend on the regular rule."""
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
    kept, taken = [_singular(6, 37)], []  # first: code, tables and scratch that every grid shares
    for nq in (1, 37):
        before = torch.cuda.mem_get_info()[0]
        kept.append(_singular(6, nq))
        assert kept[-1][1].shape == (81920, 81920)
        taken.append(before - torch.cuda.mem_get_info()[0])
    assert taken[1] <= taken[0] + 16e6


def test_values():
    assert np.array_equal(_singular(2, 6)[1].toarray(), _singular(2, 37)[1].toarray())
