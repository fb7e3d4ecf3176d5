"""Kernels that mirror half of a table or multiply by products of tables: the
mass part of a one-cell advection step, and one-cell mass applies of the 4D-6D
Kronecker kernel, against the same operator in extended precision.  On Lobatto
nodes their tables are rounded once and what remains is a walk of roundings; on
Legendre nodes they share the generic kernel's tables and are held to its error."""
import numpy as np
import pytest
import torch

import gendil_amd as G
from test_gpu_kron import KRON, SHAPES
from test_gpu_plane import PAIRS, PLANE

pytestmark = pytest.mark.gpu

LD = np.longdouble
U = 2.0**-53


def legendre(n, t):
    """P_n and P_n' at t (|t| < 1)."""
    pm, p = np.ones_like(t), t
    for k in range(1, n):
        pm, p = p, ((2 * k + 1) * t * p - k * pm) / LD(k + 1)
    return p, n * (t * p - pm) / (t * t - 1)


def rule(basis, n):
    """Points and weights on [0, 1] in extended precision; 0 Gauss-Lobatto, 1 Gauss-Legendre."""
    if basis == 1:
        t = np.cos(np.pi * (np.arange(n) + 0.75) / (n + 0.5)).astype(LD)[::-1].copy()
        for _ in range(20):
            p, dp = legendre(n, t)
            t = t - p / dp
        _, dp = legendre(n, t)
        return (1 + t) / 2, 1 / ((1 - t * t) * dp * dp)
    m = n - 1
    t = np.cos(np.pi * np.arange(1, m) / m).astype(LD)[::-1].copy()
    for _ in range(20):
        p, dp = legendre(m, t)
        t = t - dp * (1 - t * t) / (2 * t * dp - m * (m + 1) * p)
    t = np.concatenate([[LD(-1)], t, [LD(1)]])
    p = np.ones_like(t)
    p[1:-1] = legendre(m, t[1:-1])[0]
    return (1 + t) / 2, 1 / (LD(m * (m + 1)) * p * p)


def mass_matrix(basis, n, q):
    (xn, _), (xq, wq) = rule(basis, n), rule(1, q)
    B = np.array([[np.prod([(x - xn[m]) / (xn[i] - xn[m]) for m in range(n) if m != i]) for i in range(n)] for x in xq])
    return B.T @ (wq[:, None] * B)


def apply_error(op, dtype, D, n, M):
    """Largest relative 2-norm error of the apply over a few random vectors."""
    worst = 0.0
    for seed in range(4):
        x = G.fill_random(op.num_dofs, seed)
        if dtype == torch.float32:
            x = x.astype(np.float32).astype(np.float64)
        y = op(torch.as_tensor(x, dtype=dtype, device="cuda"), torch.empty(op.num_dofs, dtype=dtype, device="cuda"))
        want = x.astype(LD).reshape([n] * D)
        for _ in range(D):
            want = np.tensordot(want, M, axes=([0], [1]))
        d = y.cpu().numpy().astype(LD) - want.ravel()
        worst = max(worst, float(np.sqrt((d * d).sum() / (want * want).sum())))
    return worst


def one_cell(D, basis, n):
    fe = (G.MakeLobattoFiniteElement, G.MakeLegendreFiniteElement)[basis](n - 1)
    return G.MakeFiniteElementSpace(G.CartesianMesh([1] * D, [1.0] * D, [0.0] * D, True), fe)


@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("n,q", PAIRS)
def test_plane_kernel(n, q, basis):
    """Six 1D contractions of up to 6 products, and four more factors: with tables rounded once the roundings add up
    like a walk, sqrt(6 (6 + 1) + 4) U = 7 U.  Entries a few units off, the same in every sum, add up linearly: 8 of
    the 11 Lobatto pairs were beyond it, up to 17 U, with the tables as FP64 arithmetic gives them.  Legendre: the same
    tables in the generic kernel, the sums in another order, a walk of 2 U apart.  The advection part, 2^-80 of the
    mass, is below any rounding."""
    beta = G.fields.VectorField([G.fields.SeparableField.constant(1.0)] * 3)
    op = G.MakeMassAdvectionOperator(one_cell(3, basis, n), G.MakeIntegrationRule(q), beta, mass_coef=1.0,
                                     adv_coef=2.0**-80)
    M = mass_matrix(basis, n, q)
    bound = 7 * U
    if basis == 1:
        op.plan.set_variant(torch.float64, 0)
        bound = apply_error(op, torch.float64, 3, n, M) + 2 * U
    op.plan.set_variant(torch.float64, PLANE)
    assert apply_error(op, torch.float64, 3, n, M) <= bound


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("D,n", SHAPES)
def test_kronecker_kernel(D, n, basis, dtype):
    """D contractions of n products with a mass matrix that rounds to almost nothing, and one factor: sqrt(D n + 1) U in
    FP64 as a walk.  FP32: FP64 sums, stored (D + 1) / 2 times.  With M rounded entry by entry its error is the same in
    every value and axis.  FP64 on Legendre nodes: the generic kernel's tables, the sums in another order, a walk of
    2 U apart."""
    op = G.MakeMassFiniteElementOperator(one_cell(D, basis, n), G.MakeIntegrationRule(n), None)
    op.plan.set_variant(dtype, KRON)
    assert op.plan.query_variant(dtype, 1.0, 0.0) == KRON
    u = U if dtype == torch.float64 else 2.0**-24
    bound = (D * n + 1) ** 0.5 if dtype == torch.float64 else ((D + 1) // 2) ** 0.5
    M = mass_matrix(basis, n, n)
    err = apply_error(op, dtype, D, n, M) / u
    if basis == 1 and dtype == torch.float64:
        if (D, n) == (6, 4):
            pytest.skip("the generic kernel has no room for these elements")
        op.plan.set_variant(dtype, 0)
        bound = apply_error(op, dtype, D, n, M) / u + 2.0
    print(f"error {err:.2f} U, bound {bound:.2f} U")
    assert err <= bound
