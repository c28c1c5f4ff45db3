"""Batches whose items lie in different phase tiers, with few tiles each (which then share launches) and, for the
tier of the first items, many: every item against the oracle, 1e-12 relative."""
import numpy as np
import pytest

import oracle_lib as O
from bempp_amd.assembly.batch import BatchAssembler
from bempp_amd.assembly.boundary import BoundaryAssemblerOptions, OperatorType, create_helmholtz_assembler
from bempp_amd.element import Continuity, Family, ReferenceCellType, create_family
from bempp_amd.function_space import function_space
from bempp_amd.grid import Grid
from test_gpu_tile_parts import _torus

pytestmark = pytest.mark.gpu

OPS = {"single_layer": OperatorType.SingleLayer, "double_layer": OperatorType.DoubleLayer,
       "adjoint_double_layer": OperatorType.AdjointDoubleLayer, "hypersingular": OperatorType.Hypersingular}
FAMILY = create_family(Family.Lagrange, 0, Continuity.Discontinuous)


@pytest.mark.parametrize("ks", [(0.2, 0.5, 1.5, 9.0), (0.2, 0.5, -1.5), (0.2, 9.0), (0.5, 1.5), (0.2, 0.4), (1.5, 9.0)])
@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("nq", [3, 6, 16])
@pytest.mark.parametrize("copies", [1, 1100])
def test_tiers(ks, op, nq, copies):
    if copies > 1 and (nq != 3 or op != "single_layer"):
        pytest.skip("many tiles once")
    o = BoundaryAssemblerOptions()
    o.set_regular_quadrature_degree(ReferenceCellType.Triangle, nq)
    p, c = _torus(9, 5)  # 90 cells, three tiles of symmetric operators
    s = function_space(Grid(p, c), FAMILY)
    k = list(ks) + [ks[0]] * (copies - 1)
    A = BatchAssembler([create_helmholtz_assembler(x, OPS[op], o) for x in k], [s] * len(k)).assemble()
    for i in list(range(len(ks))) + [len(k) - 1]:
        R = O.assemble("helmholtz", op, p, c, k=k[i], nq=nq, nsing=4)
        assert np.linalg.norm(A[i].cpu().numpy() - R) <= 1e-12 * np.linalg.norm(R)
