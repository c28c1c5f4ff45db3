"""Grid.set_points drops the cached device geometry whatever the coordinates: the shape gradient that
allocates nothing is refused until an ordinary call has built it again. The backward pass of the
bilinear form takes the geometry that its own forward pass left, and sets its vertices again where
they were moved in between: gradients equal to those of a grid of its own, 1e-12 relative (order of
the additions)."""
import numpy as np
import pytest
import torch

from bempp_amd import _lib as L
from bempp_amd.assembly.boundary import OperatorType, create_laplace_assembler
from bempp_amd.autograd import bilinear_form
from test_zz_no_alloc import _dp0, _noalloc, _options, _perturbed, _vectors

pytestmark = pytest.mark.gpu


def test_same_points():
    a = create_laplace_assembler(OperatorType.SingleLayer, _options())
    g = _perturbed(1, 5)
    s = _dp0(g)
    u = _vectors(len(g.cells), np.float64, 6)
    ref = a.shape_gradient(s, s, u, u)
    for _ in range(2):
        g.set_points(g.points)
        rc, _, _ = _noalloc(a, s, u, u)
        assert rc != 0 and "allocates no device memory" in L.last_error()
        got = a.shape_gradient(s, s, u, u)
        assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("moved", [False, True])
def test_backward(moved):
    a = create_laplace_assembler(OperatorType.SingleLayer, _options())
    g = _perturbed(1, 7)
    s = _dp0(g)
    p = g.points
    u, v = (torch.from_numpy(_vectors(len(g.cells), np.float64, i)) for i in (8, 9))
    x = torch.from_numpy(p).requires_grad_()
    J = bilinear_form(x, u, v, a, s)
    if moved:
        g.set_points(1.5 * p)
    J.backward()
    ref = a.shape_gradient(*(2 * [_dp0(_perturbed(1, 7))]), u.numpy(), v.numpy())
    assert np.linalg.norm(x.grad.numpy() - ref) <= 1e-12 * np.linalg.norm(ref)
    assert np.array_equal(g.points, p)
