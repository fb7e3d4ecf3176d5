"""The 4D-6D Kronecker kernel against the CPU oracle: every compiled (dim,
nodes) with both bases and more points than nodes; one-cell axes, part-filled
last blocks; constant components, components over another axis and over their
own, of both signs and zero, given as tables or as an affine field; no and zero
inflow data; sigma with one- and two-factor terms.  What it refuses keeps the
generic kernel.  1e-12 (FP64) and 1e-5 (FP32) relative L2."""
import numpy as np
import pytest
import torch

import gendil_amd as G
import oracle
from cases import rel_l2, sigma_field
from gendil_amd.fields import SeparableField, VectorField

pytestmark = pytest.mark.gpu

KRON = 73
SHAPES = [(4, 2), (4, 3), (4, 4), (4, 5), (5, 2), (5, 3), (5, 4), (6, 2), (6, 3), (6, 4)]


def mixed_field(D):
    """Constant, zero, over another axis (both signs), over its own axis."""
    comps = [SeparableField([(1.0, {D - 1: lambda s: 0.5 + s})]), SeparableField([(-0.7, {0: lambda s: 1.0 + s * s})]),
             SeparableField([(0.4, {2: lambda s: 2.0 - s})]), SeparableField([(0.2, {}), (-1.0, {1: lambda s: 1.5 + s})]),
             SeparableField.constant(-0.3), SeparableField.constant(0.0)]
    return VectorField(comps[:D])


def phase_affine(D):
    A = np.zeros((D, D))
    for d in range(D // 2):
        A[d, D - 1 - d] = -1.0 if d == 1 else 0.8
    return G.AffineField(A, np.concatenate([np.zeros(D - 1), [0.1]]))


def run(D, n, q, basis, sizes, periodic, beta, bc, sigma, mc, ac):
    mesh = G.CartesianMesh(sizes, [0.7 / s for s in sizes], [0.05 * (d + 1) for d in range(D)], periodic)
    fe = G.MakeLobattoFiniteElement(n - 1) if basis == "L" else G.MakeLegendreFiniteElement(n - 1)
    fes, ir = G.MakeFiniteElementSpace(mesh, fe), G.MakeIntegrationRule(q)
    kw = {}
    if ac == 0.0:
        op = G.MakeMassFiniteElementOperator(fes, ir, sigma)
    else:
        op = G.MakeMassAdvectionOperator(fes, ir, beta, sigma=sigma, bc=bc, mass_coef=mc, adv_coef=ac)
        kw = dict(adv_coef=ac, adv=beta, bc=bc)
    if mc != 0.0:
        kw.update(mass_coef=mc, sigma=sigma)
    x = G.fill_random(op.num_dofs, 17)
    for dtype, tol in ((torch.float64, 1e-12), (torch.float32, 1e-5)):
        op.plan.set_variant(dtype, KRON)
        assert op.plan.query_variant(dtype, mc, ac) == KRON
        xr = x.astype(np.float32).astype(np.float64) if dtype == torch.float32 else x
        y = torch.full((op.num_dofs,), float("nan"), dtype=dtype, device="cuda")
        op(torch.as_tensor(x, dtype=dtype, device="cuda"), y)
        assert rel_l2(y.double().cpu().numpy(), oracle.Problem(fes, ir, **kw).apply(xr)) <= tol


@pytest.mark.parametrize("basis", ["L", "G"])
@pytest.mark.parametrize("D,n", SHAPES)
def test_step_every_shape(D, n, basis):
    q = n + 1 if (D, n + 1) in ((4, 3), (4, 4), (4, 5), (4, 6), (5, 3), (5, 4), (6, 3), (6, 4)) else n
    sizes = [3, 2, 2, 3, 1, 2][:D] if n > 2 else [5, 3, 2, 3, 1, 2][:D]
    run(D, n, q, basis, sizes, [d % 2 == 0 for d in range(D)], mixed_field(D), 0.0, sigma_field("poly", D), 0.6, 0.3)


@pytest.mark.parametrize("D", [4, 5, 6])
@pytest.mark.parametrize("bc", [None, 0.0])
@pytest.mark.parametrize("kind", ["mixed", "affine"])
def test_advection_boundaries_and_one_cell_axes(D, bc, kind):
    beta = mixed_field(D) if kind == "mixed" else phase_affine(D)
    run(D, 2, 3, "L", [1, 4, 1, 7, 2, 1][:D], False, beta, bc, None, 0.0, 1.0)
    run(D, 2, 3, "L", [1, 4, 1, 3, 2, 1][:D], True, beta, bc, None, 0.0, -0.5)


@pytest.mark.parametrize("D,n,sizes", [(4, 4, [5, 5, 5, 6]), (4, 4, [8, 7, 7, 8]), (4, 3, [8, 8, 8, 7]), (5, 3, [5, 4, 5, 4, 4])], ids=str)
def test_block_sizes_of_one_round(D, n, sizes):
    """Meshes whose elements per block follow the blocks that are resident at once."""
    run(D, n, n, "L", sizes, False, mixed_field(D), None, None, 0.0, 1.0)


@pytest.mark.parametrize("D,n,q", [(4, 5, 6), (5, 3, 4), (6, 3, 4)])
def test_mass(D, n, q):
    for sigma in (None, sigma_field("poly", D)):
        run(D, n, q, "G", [2, 3, 1, 2, 2, 1][:D], False, None, None, sigma, 1.0, 0.0)


def test_what_it_refuses_and_where_it_is_the_default():
    mesh = G.CartesianMesh([3] * 4, [1 / 3] * 4, [0.0] * 4, False)  # 81 elements
    fes, ir = G.MakeFiniteElementSpace(mesh, G.MakeLobattoFiniteElement(2)), G.MakeIntegrationRule(3)

    def variant(beta, bc=None, sigma=None, mc=0.0):
        op = G.MakeMassAdvectionOperator(fes, ir, beta, sigma=sigma, bc=bc, mass_coef=mc, adv_coef=1.0)
        return op.plan.query_variant(torch.float64, mc, 1.0)

    one = [SeparableField.constant(1.0)] * 3
    assert variant(mixed_field(4)) == KRON
    assert variant(mixed_field(4), bc=2.0) == 0
    assert variant(VectorField([SeparableField([(1.0, {1: lambda s: s - 0.5})])] + one)) == 0  # both signs on a face
    assert variant(VectorField([SeparableField([(1.0, {1: lambda s: s, 2: lambda s: s})])] + one)) == 0
    three = SeparableField([(1.0, {0: lambda s: s, 1: lambda s: s, 2: lambda s: s})])
    assert variant(mixed_field(4), sigma=three, mc=1.0) == 0 and variant(mixed_field(4), sigma=three) == KRON
    op = G.MakeAdvectionOperator(fes, ir, mixed_field(4))
    op.plan.set_variant(torch.float64, 0)
    assert op.plan.query_variant(torch.float64, 0.0, 1.0) == 0


def test_pinned_where_the_two_node_kernel_also_serves():
    """Order 1 with constant coefficients: the two-node kernel by default, the Kronecker kernel once pinned."""
    beta = VectorField([SeparableField.constant(c) for c in (1.0, -0.5, 0.25, 2.0)])
    run(4, 2, 2, "L", [5, 3, 2, 3], False, beta, 0.0, None, 0.6, 0.3)
    mesh = G.CartesianMesh([5, 3, 2, 3], [0.2] * 4, [0.0] * 4, False)
    op = G.MakeAdvectionOperator(G.MakeFiniteElementSpace(mesh, G.MakeLobattoFiniteElement(1)), G.MakeIntegrationRule(2), beta)
    assert op.plan.query_variant(torch.float64, 0.0, 1.0) == 64
    for variant in (KRON, 64):
        op.plan.set_variant(torch.float64, variant)
        assert op.plan.query_variant(torch.float64, 0.0, 1.0) == variant


@pytest.mark.parametrize("D,n,dtype,faster", [(4, 4, torch.float64, [5, 5, 5, 5]), (4, 5, torch.float64, [6, 6, 6, 5]),
                                              (5, 4, torch.float32, [4, 4, 4, 4, 2])], ids=str)
def test_mass_alone_with_few_points(D, n, dtype, faster):
    """Mass applies with q = n that the generic kernel does faster keep it: below or above 1,000 elements."""
    slower = [6, 6, 6, 5] if faster[0] == 5 else [6, 6, 6, 5, 1] if D == 5 else [4] * 4
    for sizes, sigma, want in ((faster, "poly", KRON), (slower, "poly", 0), (slower, "one", KRON)):
        fes = G.MakeFiniteElementSpace(G.CartesianMesh(sizes, [1 / s for s in sizes], [0.0] * D, False), G.MakeLobattoFiniteElement(n - 1))
        op = G.MakeMassFiniteElementOperator(fes, G.MakeIntegrationRule(n), sigma_field("poly", D) if sigma == "poly" else None)
        assert op.plan.query_variant(dtype, 1.0, 0.0) == want
