"""Helmholtz operators at small wavenumbers, where quantities scaled by |k| leave their type's range:
mixed precision (single and batched) against FP64, all operators: 1e-6 relative in the norm as for
every mixed-precision operator, all entries finite; potentials, P1 and quadrilateral operators in
FP64 against the Laplace ones, whose values they have up to a relative |k| times the meshes'
extent: 1e-12 for |k| <= 1e-13."""
import numpy as np
import pytest
import torch

import oracle_lib as O
import quad_meshes as M
from bempp_amd.assembly.batch import BatchAssembler
from bempp_amd.assembly.boundary import (BoundaryAssemblerOptions, OperatorType, Precision, create_helmholtz_assembler,
                                         create_laplace_assembler)
from bempp_amd.assembly.potential import create_helmholtz_potential_assembler
from bempp_amd.element import Continuity, Family, ReferenceCellType, create_family
from bempp_amd.function_space import function_space
from bempp_amd.grid import Grid
from test_gpu_tile_parts import _torus

pytestmark = pytest.mark.gpu


def _options(nq=6, precision=Precision.FP64):
    o = BoundaryAssemblerOptions()
    o.set_regular_quadrature_degree(ReferenceCellType.Quadrilateral, 16)
    o.set_regular_quadrature_degree(ReferenceCellType.Triangle, nq)
    o.set_precision(precision)
    return o


def _space(g, degree, continuity=Continuity.Standard):
    return function_space(g, create_family(Family.Lagrange, degree, continuity if degree else Continuity.Discontinuous))


def _thin_torus():
    """2304 cells in 36 tiles, most of them very far from each other (tube radius 0.1)."""
    p, c = _torus(96, 12)
    ring = p * [1, 1, 0]
    ring /= np.linalg.norm(ring, axis=1, keepdims=True)
    return ring + 0.25 * (p - ring), c


@pytest.mark.parametrize("k", [1e-2, 1e-3, -1e-4, 1e-5, 1e-6, 1e-8, 1e-12, 1e-20, 1e-40])
@pytest.mark.parametrize("op", list(OperatorType)[:4])
@pytest.mark.parametrize("nq", [6, 7])
def test_mixed(k, op, nq):
    p, c = _thin_torus()
    s = _space(Grid(p, c), 0)
    R = create_helmholtz_assembler(k, op, _options(nq)).assemble_device(s, s)
    a = [create_helmholtz_assembler(x, op, _options(nq, Precision.Mixed)) for x in (k, 2.0 * k)]
    A = a[0].assemble_device(s, s)
    B = BatchAssembler(a, [s, s]).assemble()[0]
    for x in (A, B):
        assert torch.isfinite(torch.view_as_real(x)).all()
        assert torch.linalg.norm(x - R) <= 1e-6 * torch.linalg.norm(R)


@pytest.mark.parametrize("scale", [1.0, 1e-4])
@pytest.mark.parametrize("k", [0.0, 1e-16, -1e-90, 1e-99, 2e-100, 1e-160, 1e-300])
@pytest.mark.parametrize("op", ["single_layer", "double_layer"])
@pytest.mark.parametrize("degree", [0, 1])
@pytest.mark.parametrize("nq", [3, 6, 16])
def test_potential(scale, k, op, degree, nq):
    p, c = O.sphere(1, "icosahedron")
    rng = np.random.default_rng(nq)
    x = rng.standard_normal((70, 3))
    x *= scale * (rng.uniform(1.1, 8.0, 70) / np.linalg.norm(x, axis=1))[:, None]
    p = scale * p
    kind = OperatorType.SingleLayer if op == "single_layer" else OperatorType.DoubleLayer
    got = create_helmholtz_potential_assembler(k, kind, _options(nq)).assemble(_space(Grid(p, c), degree), x)
    R = O.potential("laplace", op, p, c, x, space=(degree, degree == 1), nq=nq)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - R) <= 1e-12 * np.linalg.norm(R)


@pytest.mark.parametrize("scale", [1.0, 1e-4])
@pytest.mark.parametrize("k", [0.0, 1e-16, -1e-90, 1e-99, 2e-100, 1e-160, 1e-300])
@pytest.mark.parametrize("op", [OperatorType.SingleLayer, OperatorType.DoubleLayer, OperatorType.AdjointDoubleLayer])
@pytest.mark.parametrize("degree,nq", [(0, 6), (0, 16), (1, 3), (1, 16)])
def test_dense(scale, k, op, degree, nq):
    p, c = _torus(9, 7)
    s = _space(Grid(scale * p, c), degree)
    got = create_helmholtz_assembler(k, op, _options(nq)).assemble(s, s)
    R = create_laplace_assembler(op, _options(nq)).assemble(s, s)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - R) <= 1e-12 * np.linalg.norm(R)


@pytest.mark.parametrize("scale", [1.0, 1e-4])
@pytest.mark.parametrize("k", [0.0, 1e-16, -1e-90, 1e-160, 1e-300])
@pytest.mark.parametrize("op", [OperatorType.SingleLayer, OperatorType.DoubleLayer])
def test_quadrilaterals(scale, k, op):
    p, c = M.cubed_sphere(4)
    s = _space(Grid(scale * p, c), 0)
    got = create_helmholtz_assembler(k, op, _options()).assemble(s, s)
    R = create_laplace_assembler(op, _options()).assemble(s, s)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - R) <= 1e-12 * np.linalg.norm(R)
