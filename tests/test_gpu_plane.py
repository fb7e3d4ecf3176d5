"""The plane kernel (uniform 3D apply for any basis, rule and separable or
affine field) against the CPU oracle.

Sizes: one cell, one-cell axes (periodic: an element is its own neighbour), a
mesh smaller than a block, meshes whose last block is partly filled.  Every
compiled (nodes, points) pair, both bases, both precisions; fields over one,
two and three coordinates, fields whose sign changes within a face, affine
fields; no, zero and polynomial inflow data.  Tolerances as for every other
kernel: 1e-12 (FP64) and 1e-5 (FP32) relative L2."""
import numpy as np
import pytest
import torch

import gendil_amd as G
import oracle
from cases import TWO_PI, bc_field, beta_field, diffusivity_field, rel_l2, sigma_field
from gendil_amd.fields import SeparableField, VectorField

pytestmark = pytest.mark.gpu

PLANE = 72
PAIRS = [(2, 2), (2, 3), (2, 4), (3, 3), (3, 4), (3, 5), (4, 4), (4, 5), (4, 6), (5, 5), (5, 6)]


def field(kind):
    if kind == "mixed":  # rank 2 and 3, one to three coordinates, both signs within a face
        return VectorField([
            SeparableField([(0.3, {}), (1.0, {1: lambda s: np.sin(TWO_PI * s), 2: lambda s: np.cos(TWO_PI * s)})]),
            SeparableField([(-0.2, {0: lambda s: s}), (0.7, {0: lambda s: np.cos(TWO_PI * s), 1: lambda s: s,
                                                             2: lambda s: 1.0 - s}), (0.1, {2: lambda s: s})]),
            SeparableField([(1.0, {0: lambda s: 0.4 - s})]),
        ])
    if kind == "affine":
        return G.AffineField(np.array([[0.3, -1.0, 0.2], [0.9, 0.1, -0.4], [-0.5, 0.6, 0.7]]), np.array([0.1, -0.2, 0.05]))
    return beta_field(kind, 3)


def space(sizes, p, basis, periodic):
    h = [0.9 / s * (1.0 + 0.2 * d) for d, s in enumerate(sizes)]
    mesh = G.CartesianMesh(sizes, h, [0.1, -0.2, 0.3], periodic)
    fe = G.MakeLobattoFiniteElement(p) if basis == "L" else G.MakeLegendreFiniteElement(p)
    return G.MakeFiniteElementSpace(mesh, fe)


def check(fes, q, dtype, beta, bc, sigma, mc, ac):
    ir = G.MakeIntegrationRule(q)
    g = bc_field(bc, 3)
    if ac == 0.0:
        op = G.MakeMassFiniteElementOperator(fes, ir, sigma)
        kw = {}
    else:
        op = G.MakeMassAdvectionOperator(fes, ir, beta, sigma=sigma, bc=g, mass_coef=mc, adv_coef=ac)
        kw = dict(adv_coef=ac, adv=beta, bc=g)
    op.plan.set_variant(dtype, PLANE)
    assert op.plan.query_variant(dtype, mc, ac) == PLANE
    x = G.fill_random(op.num_dofs, 11)
    y = torch.full((op.num_dofs,), float("nan"), dtype=dtype, device="cuda")
    op(torch.as_tensor(x, dtype=dtype, device="cuda"), y)
    if mc != 0.0:
        kw.update(mass_coef=mc, sigma=sigma)
    xr = x.astype(np.float32).astype(np.float64) if dtype == torch.float32 else x
    ref = oracle.Problem(fes, ir, **kw).apply(xr)
    assert rel_l2(y.double().cpu().numpy(), ref) <= (1e-12 if dtype == torch.float64 else 1e-5)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("basis", ["L", "G"])
@pytest.mark.parametrize("n,q", PAIRS)
def test_step_every_pair(n, q, basis, dtype):
    fes = space((5, 3, 4), n - 1, basis, [True, False, True])
    check(fes, q, dtype, field("mixed"), "poly", sigma_field("poly", 3), 0.7, 0.4)


@pytest.mark.parametrize("sizes", [(1, 1, 1), (1, 5, 1), (7, 1, 2), (33, 1, 1), (13, 11, 17)], ids=str)
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("kind,bc", [("mixed", "none"), ("affine", "zero"), ("affine", "poly"), ("const", "poly")])
def test_advection_sizes_and_boundaries(sizes, periodic, kind, bc):
    check(space(sizes, 2, "L", periodic), 4, torch.float64, field(kind), bc, None, 0.0, 1.0)


@pytest.mark.parametrize("n,q", [(4, 6), (5, 5), (5, 6)])
@pytest.mark.parametrize("sizes", [(13, 11, 12), (13, 11, 17), (19, 17, 13), (25, 21, 20)], ids=str)
def test_block_sizes_of_one_round(n, q, sizes):
    """Meshes whose elements per block follow the blocks that are resident at once: 4, 5, 9 and 21 elements."""
    check(space(sizes, n - 1, "L", [False, True, False]), q, torch.float64, field("mixed"), "none", None, 0.0, 1.0)


@pytest.mark.parametrize("n,q", [(2, 4), (3, 5), (4, 6), (5, 6)])
@pytest.mark.parametrize("sizes", [(1, 1, 1), (9, 5, 3)], ids=str)
def test_mass(n, q, sizes):
    for dtype in (torch.float64, torch.float32):
        check(space(sizes, n - 1, "G", False), q, dtype, None, "none", sigma_field("poly", 3), 1.0, 0.0)


def test_default_where_no_faster_kernel_serves():
    """The plane kernel is the default for rules, bases and fields that the Kronecker and register kernels refuse;
    0 pins the generic kernel."""
    fes = space((6, 5, 4), 3, "L", False)
    op = G.MakeAdvectionOperator(fes, G.MakeIntegrationRule(5), field("mixed"))
    assert op.plan.query_variant(torch.float64, 0.0, 1.0) == PLANE
    op.plan.set_variant(torch.float64, 0)
    assert op.plan.query_variant(torch.float64, 0.0, 1.0) == 0
    x = torch.as_tensor(G.fill_random(op.num_dofs, 2), device="cuda")
    generic = op(x, torch.empty_like(x)).cpu().numpy()
    op.plan.set_variant(torch.float64, -1)
    assert rel_l2(op(x, torch.empty_like(x)).cpu().numpy(), generic) <= 1e-13


DIFF_PAIRS = [(2, 3), (2, 4), (3, 3), (3, 4), (3, 5), (4, 4), (4, 5), (4, 6)]


def check_diffusion(fes, q, dtype, mu, sigma, kappa):
    ir = G.MakeIntegrationRule(q)
    op = G.MakeDiffusionOperator(fes, ir, mu, sigma, kappa)
    x = G.fill_random(op.num_dofs, 13)
    y = torch.full((op.num_dofs,), float("nan"), dtype=dtype, device="cuda")
    op(torch.as_tensor(x, dtype=dtype, device="cuda"), y)
    xr = x.astype(np.float32).astype(np.float64) if dtype == torch.float32 else x
    ref = oracle.Problem(fes, ir).diffusion(xr, mu, sigma, kappa)
    assert rel_l2(y.double().cpu().numpy(), ref) <= (1e-12 if dtype == torch.float64 else 1e-5)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("basis", ["L", "G"])
@pytest.mark.parametrize("n,q", DIFF_PAIRS)
def test_diffusion_every_pair(n, q, basis, dtype):
    """The diffusion plane kernel, an eight-term diffusivity, mixed boundaries; small meshes in FP64 go to the
    generic kernel from q = 4 on."""
    for sizes in ((5, 3, 4), (17, 13, 12)):
        check_diffusion(space(sizes, n - 1, basis, [True, False, True]), q, dtype, diffusivity_field("trig", 3), -1.0, 9.0)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("sizes", [(1, 1, 1), (1, 5, 1), (33, 1, 1), (13, 11, 7), (2501, 1, 1), (1, 49, 53)], ids=str)
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("rank", [0, 1, 2, 3])
def test_diffusion_sizes_ranks_and_boundaries(sizes, periodic, rank, dtype):
    terms = [(1.5, {}), (0.3, {0: lambda s: s, 2: lambda s: 1.0 + s}), (0.2, {1: lambda s: s * s})][:rank]
    check_diffusion(space(sizes, 3, "L", periodic), 5, dtype, SeparableField(terms), 1.0 if rank == 2 else 0.0, 4.0)


def pointwise_problem(fes, q, seed):
    """Random per-point field (both signs on every face) as host arrays and as an operator."""
    rng = np.random.default_rng(seed)
    cell = rng.standard_normal((fes.mesh.num_cells, 3, q ** 3))
    faces = [rng.standard_normal((f, q * q)) for f in G.face_counts(fes.mesh)]
    dev = [torch.as_tensor(t, device="cuda") for t in (cell, *faces)]
    return cell, faces, dev


@pytest.mark.parametrize("sizes,periodic,bc", [((5, 3, 4), [True, False, True], "poly"), ((1, 1, 1), False, "zero"),
                                               ((1, 5, 1), True, "none"), ((7, 5, 3), False, "none")], ids=str)
@pytest.mark.parametrize("basis", ["L", "G"])
@pytest.mark.parametrize("n,q", PAIRS)
def test_pointwise_forward_transpose_and_gradient(n, q, basis, sizes, periodic, bc):
    """The plane kernels of the per-point field: apply, adjoint and field gradient."""
    fes = space(sizes, n - 1, basis, periodic)
    ir, g = G.MakeIntegrationRule(q), bc_field(bc, 3)
    cell, faces, dev = pointwise_problem(fes, q, 7)
    op = G.MakeAdvectionOperator(fes, ir, G.PointwiseField(dev[0], dev[1:]), g)
    u, r = G.fill_random(op.num_dofs, 21), G.fill_random(op.num_dofs, 22)
    P = oracle.Problem(fes, ir, adv_coef=1.0, adv=(cell, faces), bc=g)
    du, dr = torch.as_tensor(u, device="cuda"), torch.as_tensor(r, device="cuda")
    nan = lambda t: torch.full_like(t, float("nan"))  # noqa: E731
    y = op(du, nan(du))
    assert rel_l2(y.cpu().numpy(), P.apply(u)) <= 1e-12
    z = op.transpose(dr, nan(dr))
    assert rel_l2(z.cpu().numpy(), P.apply_transpose(r)) <= 1e-12
    dcell, dfaces = nan(dev[0]), [nan(t) for t in dev[1:]]
    op.plan.grad_beta(0.7, du, dr, dcell, dfaces)
    ref_cell, ref_faces = P.grad_beta(u, r, G.face_counts(fes.mesh))
    assert rel_l2(dcell.cpu().numpy().ravel(), 0.7 * np.asarray(ref_cell).ravel()) <= 1e-12
    for a in range(3):
        want = 0.7 * np.asarray(ref_faces[a]).ravel()
        got = dfaces[a].cpu().numpy().ravel()
        assert np.linalg.norm(got - want) <= 1e-12 * max(np.linalg.norm(want), 1e-300)


def test_pointwise_transpose_with_mass():
    fes = space((4, 3, 5), 3, "L", [False, True, False])
    ir = G.MakeIntegrationRule(5)
    cell, faces, dev = pointwise_problem(fes, 5, 9)
    sigma = sigma_field("poly", 3)
    op = G.MakeMassAdvectionOperator(fes, ir, G.PointwiseField(dev[0], dev[1:]), sigma=sigma, mass_coef=0.6, adv_coef=-0.3)
    r = G.fill_random(op.num_dofs, 5)
    z = op.transpose(torch.as_tensor(r, device="cuda"), torch.empty(op.num_dofs, dtype=torch.float64, device="cuda"))
    P = oracle.Problem(fes, ir, mass_coef=0.6, adv_coef=-0.3, sigma=sigma, adv=(cell, faces))
    assert rel_l2(z.cpu().numpy(), P.apply_transpose(r)) <= 1e-12


def pole(s):
    with np.errstate(divide="ignore"):
        return 1.0 / (s * (1.0 - s))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("basis", ["L", "G"])
@pytest.mark.parametrize("mc", [0.0, 0.7])
def test_field_infinite_on_skipped_boundary_faces(mc, basis, dtype):
    """Without boundary data a boundary face carries no flux, whatever the field is there: a component with a pole on
    its own axis's ends leaves a finite result."""
    fe = G.MakeLobattoFiniteElement(2) if basis == "L" else G.MakeLegendreFiniteElement(2)
    fes = G.MakeFiniteElementSpace(G.CartesianMesh([4, 2, 4], [0.25, 0.5, 0.25], [0.0] * 3, False), fe)
    beta = VectorField([SeparableField([(0.1 * (d + 1), {d: pole})]) for d in range(3)])
    check(fes, 4, dtype, beta, "none", None, mc, 1.0)


def test_pointwise_field_unset_on_skipped_boundary_faces():
    """The boundary rows of a per-point field are not used without boundary data: NaN there reaches neither the apply nor
    the transpose, and the gradient is 0 there."""
    sizes, n, q = (3, 4, 5), 3, 4
    fes, ir = space(sizes, n - 1, "L", False), G.MakeIntegrationRule(q)
    cell, faces, _ = pointwise_problem(fes, q, 3)
    edge = []
    for a in range(3):
        ext = [s + (d == a) for d, s in enumerate(sizes)]
        at = np.indices(ext[::-1]).reshape(3, -1)[2 - a]
        edge.append((at == 0) | (at == sizes[a]))
        faces[a][edge[a]] = np.nan
    dev = [torch.as_tensor(t, device="cuda") for t in (cell, *faces)]
    op = G.MakeAdvectionOperator(fes, ir, G.PointwiseField(dev[0], dev[1:]))
    u, r = G.fill_random(op.num_dofs, 21), G.fill_random(op.num_dofs, 22)
    P = oracle.Problem(fes, ir, adv_coef=1.0, adv=(cell, faces))
    du, dr = torch.as_tensor(u, device="cuda"), torch.as_tensor(r, device="cuda")
    assert rel_l2(op(du, torch.empty_like(du)).cpu().numpy(), P.apply(u)) <= 1e-12
    assert rel_l2(op.transpose(dr, torch.empty_like(dr)).cpu().numpy(), P.apply_transpose(r)) <= 1e-12
    dcell, dfaces = torch.empty_like(dev[0]), [torch.empty_like(t) for t in dev[1:]]
    op.plan.grad_beta(1.0, du, dr, dcell, dfaces)
    for a in range(3):
        g = dfaces[a].cpu().numpy()
        assert np.all(g[edge[a]] == 0.0) and np.all(np.isfinite(g))


def test_nan_in_a_pointwise_face_field_reaches_the_transpose():
    """NaN at a point of one inner face per axis: NaN in both elements of the face, nowhere else."""
    sizes, n, q = (5, 3, 4), 3, 4
    fes, ir = space(sizes, n - 1, "G", True), G.MakeIntegrationRule(q)
    for a in range(3):
        cell, faces, _ = pointwise_problem(fes, q, 4)
        faces[a][2 + 5 * 2 + 15 * 2, 7] = np.nan
        dev = [torch.as_tensor(t, device="cuda") for t in (cell, *faces)]
        op = G.MakeAdvectionOperator(fes, ir, G.PointwiseField(dev[0], dev[1:]))
        r = G.fill_random(op.num_dofs, 22)
        dr = torch.as_tensor(r, device="cuda")
        got = op.transpose(dr, torch.empty_like(dr)).cpu().numpy()
        want = oracle.Problem(fes, ir, adv_coef=1.0, adv=(cell, faces)).apply_transpose(r)
        assert np.isnan(want).sum() == 2 * n**3
        assert np.array_equal(np.isnan(got), np.isnan(want))


@pytest.mark.parametrize("n,q", PAIRS)
def test_nan_in_a_pointwise_boundary_field_gives_no_outflow(n, q):
    """NaN at a point of one boundary face per axis, with data: the transpose takes it as no outflow."""
    fes, ir = space((5, 3, 4), n - 1, "G", False), G.MakeIntegrationRule(q)
    cell, faces, _ = pointwise_problem(fes, q, 4)
    for a, f in enumerate((5, 3 * 5, 4 * 15)):  # an upper boundary face
        faces[a][f, 1] = np.nan
    dev = [torch.as_tensor(t, device="cuda") for t in (cell, *faces)]
    op = G.MakeAdvectionOperator(fes, ir, G.PointwiseField(dev[0], dev[1:]), bc_field("poly", 3))
    r = G.fill_random(op.num_dofs, 22)
    dr = torch.as_tensor(r, device="cuda")
    got = op.transpose(dr, torch.empty_like(dr)).cpu().numpy()
    for f in faces:
        f[np.isnan(f)] = 0.0
    want = oracle.Problem(fes, ir, adv_coef=1.0, adv=(cell, faces), bc=bc_field("poly", 3)).apply_transpose(r)
    assert rel_l2(got, want) <= 1e-12


def pinned(op, dtype, run):
    """run() by default and with the generic kernel pinned: other sums, so other last bits."""
    default = run()
    op.plan.set_variant(dtype, 0)
    generic = run()
    op.plan.set_variant(dtype, -1)
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    for a, b in zip(default, generic):
        assert not torch.equal(a, b) and rel_l2(a.double().cpu().numpy(), b.double().cpu().numpy()) <= tol
    assert all(torch.equal(a, b) for a, b in zip(default, run()))


@pytest.mark.parametrize("bc", ["none", "poly"])
@pytest.mark.parametrize("basis", ["L", "G"])
@pytest.mark.parametrize("n,q", PAIRS)
def test_pinned_generic_kernels_of_the_pointwise_field(n, q, basis, bc):
    fes = space((4, 5, 3), n - 1, basis, [False, True, False])
    _, _, dev = pointwise_problem(fes, q, 7)
    op = G.MakeAdvectionOperator(fes, G.MakeIntegrationRule(q), G.PointwiseField(dev[0], dev[1:]), bc_field(bc, 3))
    u, r = (torch.as_tensor(G.fill_random(op.num_dofs, s), device="cuda") for s in (21, 22))

    def run():
        dcell, dfaces = torch.empty_like(dev[0]), [torch.empty_like(t) for t in dev[1:]]
        op.plan.grad_beta(0.7, u, r, dcell, dfaces)
        return [op.transpose(r, torch.empty_like(r)), dcell, *dfaces]

    pinned(op, torch.float64, run)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("n,q", DIFF_PAIRS)
def test_pinned_generic_kernel_of_the_diffusion(n, q, dtype):
    fes = space((17, 13, 12), n - 1, "G", [True, False, True])
    op = G.MakeDiffusionOperator(fes, G.MakeIntegrationRule(q), diffusivity_field("trig", 3), -1.0, 9.0)
    x = torch.as_tensor(G.fill_random(op.num_dofs, 13), dtype=dtype, device="cuda")
    pinned(op, dtype, lambda: [op(x, torch.empty_like(x))])
