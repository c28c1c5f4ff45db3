"""Potentials on meshes in random cell order, where a cell's DOFs lie in different blocks, on both sides of
the rules by which the cells are taken by DOF blocks or once: against the oracle, 1e-12 relative."""
import numpy as np
import pytest

import oracle_lib as O
from bempp_amd.assembly.boundary import BoundaryAssemblerOptions, OperatorType
from bempp_amd.assembly.potential import create_helmholtz_potential_assembler, create_laplace_potential_assembler
from bempp_amd.element import Continuity, Family, ReferenceCellType, create_family
from bempp_amd.function_space import function_space
from bempp_amd.grid import Grid
from test_gpu_tile_parts import _torus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu,nv", [(13, 5), (31, 17)])  # 65 and 527 DOFs
@pytest.mark.parametrize("points", [50, 1500])
@pytest.mark.parametrize("k", [None, 3.0])
@pytest.mark.parametrize("op", ["single_layer", "double_layer"])
@pytest.mark.parametrize("nq", [3, 6, 16, 37])
def test_shuffled(nu, nv, points, k, op, nq):
    p, c = _torus(nu, nv)
    rng = np.random.default_rng(nq)
    c = c[rng.permutation(len(c))]
    x = rng.standard_normal((points, 3))
    x *= (rng.uniform(3.0, 8.0, points) / np.linalg.norm(x, axis=1))[:, None]
    o = BoundaryAssemblerOptions()
    o.set_regular_quadrature_degree(ReferenceCellType.Triangle, nq)
    kind = OperatorType.SingleLayer if op == "single_layer" else OperatorType.DoubleLayer
    a = (create_laplace_potential_assembler(kind, o) if k is None else
         create_helmholtz_potential_assembler(k, kind, o))
    s = function_space(Grid(p, c), create_family(Family.Lagrange, 1, Continuity.Standard))
    R = O.potential("laplace" if k is None else "helmholtz", op, p, c, x, space=(1, True), k=k or 0.0, nq=nq)
    assert np.linalg.norm(a.assemble(s, x) - R) <= 1e-12 * np.linalg.norm(R)
