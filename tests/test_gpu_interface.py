"""The one-wave interface kernel (conforming 3D interfaces of two meshes whose
orders and bases may differ) against the CPU oracle, accumulated into a random
y: every face, one face, face counts that leave the last wave part-filled, the
smallest and largest nodes and points of its range, rules of one face and of
many faces per wave.  1e-12 relative L2, as for every FP64 kernel."""
import numpy as np
import pytest
import torch

import gendil_amd as G
import oracle
from cases import beta_field, beta_numpy, rel_l2

pytestmark = pytest.mark.gpu


def check(face, sizes, n, bases, q, coef):
    axis, up = face % 3, face >= 3
    h = [0.3, 0.2, 0.25]
    other = list(sizes)
    other[axis] = 2
    o_minus = [0.1, -0.2, 0.3]
    o_plus = list(o_minus)
    o_plus[axis] += h[axis] * (sizes[axis] if up else -other[axis])
    make = {"L": G.MakeLobattoFiniteElement, "G": G.MakeLegendreFiniteElement}
    fm = G.MakeFiniteElementSpace(G.CartesianMesh(sizes, h, o_minus), make[bases[0]](n[0] - 1))
    fp = G.MakeFiniteElementSpace(G.CartesianMesh(other, h, o_plus), make[bases[1]](n[1] - 1), G.L2Restriction(fm.num_dofs))
    op = G.MakeAdvectionFaceOperator(fm, fp, G.CartesianIntermeshFaceConnectivity(3, face, sizes, other),
                                     G.MakeIntegrationRule(q), beta_field(coef, 3))
    N, nm = fm.num_dofs + fp.num_dofs, fm.num_dofs
    x, y0 = G.fill_random(N, 3), G.fill_random(N, 4)
    y = op(torch.as_tensor(x, device="cuda"), torch.as_tensor(y0, device="cuda"))
    want = y0.copy()
    side = lambda s, o, k, b: dict(sizes=s, h=h, origin=o, n=k, basis="LG".index(b))  # noqa: E731
    oracle.intermesh_operator(face, q, side(sizes, o_minus, n[0], bases[0]), side(other, o_plus, n[1], bases[1]),
                              beta_numpy(coef, 3), x[:nm], x[nm:], want[:nm], want[nm:])
    assert rel_l2(y.cpu().numpy() - y0, want - y0) <= 1e-12


@pytest.mark.parametrize("face", range(6))
@pytest.mark.parametrize("n,q", [((2, 4), 5), ((4, 2), 4), ((1, 3), 2)], ids=str)
def test_every_face(face, n, q):
    check(face, [3, 5, 4], n, "LL", q, "trig")


@pytest.mark.parametrize("bases", ["LG", "GL", "GG"])
@pytest.mark.parametrize("n,q", [((8, 8), 8), ((1, 1), 2), ((8, 1), 3), ((3, 5), 1), ((2, 3), 7)], ids=str)
def test_range_of_orders_and_rules(bases, n, q):
    check(4, [2, 1, 3], n, bases, q, "yzx")


@pytest.mark.parametrize("sizes", [(1, 1, 1), (9, 2, 7), (1, 1, 65)], ids=str)
def test_face_counts(sizes):
    check(1, list(sizes), (3, 2), "LL", 3, "c2")


@pytest.mark.parametrize("thick", [1, 2])
@pytest.mark.parametrize("basis,n", [("L", 1), ("G", 2), ("L", 3), ("G", 4)])
@pytest.mark.parametrize("face", [0, 2, 4])
def test_space_glued_to_itself(face, basis, n, thick):
    """One space on both sides, closing the face's axis: with one cell along it both sides are the same element, whose
    values both shares are added to."""
    sizes, h, origin, q = [5, 4, 7], [0.3, 0.2, 0.25], [0.1, -0.2, 0.3], max(n, 2)
    sizes[face % 3] = thick
    make = G.MakeLobattoFiniteElement if basis == "L" else G.MakeLegendreFiniteElement
    fes = G.MakeFiniteElementSpace(G.CartesianMesh(sizes, h, origin), make(n - 1))
    op = G.MakeAdvectionFaceOperator(fes, fes, G.CartesianIntermeshFaceConnectivity(3, face, sizes, sizes),
                                     G.MakeIntegrationRule(q), beta_field("trig", 3))
    x, y0 = G.fill_random(fes.num_dofs, 3), G.fill_random(fes.num_dofs, 4)
    y = op(torch.as_tensor(x, device="cuda"), torch.as_tensor(y0, device="cuda"))
    side = dict(sizes=sizes, h=h, origin=origin, n=n, basis="LG".index(basis))
    want = y0.copy()
    oracle.intermesh_operator(face, q, side, side, beta_numpy("trig", 3), x, x, want, want)
    # y itself, not what was added: the two shares of an order-0 element cancel.  Two additions round y twice (2e-16);
    # a lost share is of the size of y.
    assert rel_l2(y.cpu().numpy(), want) <= 1e-12
    if n > 1:
        assert rel_l2(y.cpu().numpy() - y0, want - y0) <= 1e-12
