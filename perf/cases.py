"""Performance cases: what programs built on gendil_amd have it do.

Each case is one pass through public entry points:

  transport  op(x, y) of a mass, advection or mass + advection operator on a
             uniform space (2D..6D, any compiled order and rule, FP64 / FP32)
  adjoint    advection_apply and its backward with a per-point field
  diffusion  op(x, y) of the SIPDG diffusion operator
  padaptive  op(x, y) of advection on a space with per-element orders
  coupled    two blocks of different order and the interface operator between
             them, all in one vector
  faces      the face-centric operator over a mesh's interior faces
  solve      a Krylov solve of the implicit step or of the mass matrix

exact() restates every one of them in 64 bits with plain torch, from the weak
form on the tensor rule: no code of this package takes part in it.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import gendil_amd as G

TWO_PI = 2.0 * math.pi
DEVICE = "cuda"


# ---------------------------------------------------------------------------
# fields: sums of (scale, {axis: factor}); the factors take numpy arrays (the
# package tabulates them) and torch tensors (exact() evaluates them)
# ---------------------------------------------------------------------------

def _sin(k=1, phase=0.0):
    return lambda s: (torch.sin if isinstance(s, torch.Tensor) else np.sin)(TWO_PI * (k * s + phase))


def _cos(k=1, phase=0.0):
    return lambda s: (torch.cos if isinstance(s, torch.Tensor) else np.cos)(TWO_PI * (k * s + phase))


def _id(s):
    return s


def _beta_terms(kind, D):
    """One list of terms per component."""
    if kind == "c2":  # the benchmark field (3D): one coordinate each, one sign
        return [[(1.0, {1: lambda s: 1.0 + 0.5 * _sin()(s)})], [(1.0, {2: lambda s: 0.5 + 0.5 * _cos()(s)})],
                [(1.0, {0: lambda s: 0.25 + 0.25 * _sin()(s)})]]
    if kind == "rotating":  # one coordinate each, signs change inside the mesh
        return [[(1.0, {1: lambda s: 0.5 - s})], [(1.0, {0: lambda s: s - 0.5})]] + [[(0.25, {})] for _ in range(D - 2)]
    if kind == "bubble":  # GenDiL's advection tests: beta_d = -x_d (1 - x_d)
        return [[(1.0, {d: lambda s: -s * (1.0 - s)})] for d in range(D)]
    if kind == "swirl":  # products over two coordinates
        return [[(1.0 / 2 ** d, {}), (0.5 / 2 ** d, {(d + 1) % D: _sin(), (d + 2) % D: _cos()})] for d in range(D)]
    if kind == "trig":  # GenDiL's harness field
        return [[(1.0, {(d + 1) % D: lambda s: 0.5 + _sin()(s)})] for d in range(D)]
    if kind == "const":
        return [[((-0.5) ** d, {})] for d in range(D)]
    if kind == "phase":  # D/2 space and D/2 velocity axes: beta = (v, a)
        H = D // 2
        return [[(1.0, {H + d: _id})] for d in range(H)] + [[(0.1, {})]] + [[] for _ in range(H - 1)]
    raise ValueError(kind)


def _sigma_terms(kind, D):
    if kind == "one":
        return [(1.0, {})]
    return [(1.0, {}), (1.0, {0: _id, 1: _id}), (1.0, {D - 1: lambda s: s * s})]  # 1 + x y + z^2


def _mu_terms(kind, D):
    if kind == "one":
        return [(1.0, {})]
    if D == 3:
        # 2 + 0.25 sin 2 pi x + 0.17 cos 2 pi (2y + 0.13) + 0.11 sin 2 pi (3z + 0.37)
        # + 0.07 sin 2 pi (x + 2y + 3z)
        return [(2.0, {}), (0.25, {0: _sin()}), (0.17, {1: _cos(2, 0.13)}), (0.11, {2: _sin(3, 0.37)}),
                (0.07, {0: _sin(1), 1: _cos(2), 2: _cos(3)}), (0.07, {0: _cos(1), 1: _sin(2), 2: _cos(3)}),
                (0.07, {0: _cos(1), 1: _cos(2), 2: _sin(3)}), (-0.07, {0: _sin(1), 1: _sin(2), 2: _sin(3)})]
    return [(2.0, {})] + [(0.25 / (d + 1), {d: _sin(d + 1, 0.13 * d)}) for d in range(D)]


BC_INFLOW_TERMS = [(1.0, {}), (1.0, {0: _id}), (-0.5, {1: _id})]  # g = 1 + x - 0.5 y


def _field(terms):
    return G.SeparableField([t for t in terms if t[0] != 0.0])


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def _transport(mesh, p, q, basis="gll", field="c2", bc="periodic", dtype="f64", op="advection", sigma="one"):
    return {"kind": "transport", "mesh": mesh, "p": p, "q": q, "basis": basis, "field": field, "bc": bc,
            "dtype": dtype, "op": op, "sigma": sigma}


def listed():
    return [
        # one implicit-step operator apply on a tiny mesh: a unit test, a coarse
        # level or a debugging run; the time of a call
        dict(_transport("6x6x6", 3, 4, bc="zero", op="step"), name="step_6_p3"),
        # the mass apply on an ordinary mesh (GenDiL's mass benchmark, q = n)
        dict(_transport("32x32x32", 3, 4, bc="none", op="mass"), name="mass_32_p3"),
        # over-integrated mass with a variable coefficient on ragged odd sizes in
        # FP32 (GenDiL's mass tests: q = p + 3, sigma = 1 + x y + z^2)
        dict(_transport("43x37x29", 2, 5, bc="none", op="mass", sigma="poly", dtype="f32"), name="mass_43x37x29_p2q5_f32"),
        # the headline: upwind advection, periodic, 16.8 M unknowns
        dict(_transport("64x64x64", 3, 4), name="adv_64_p3"),
        # over-integrated advection (GenDiL's range benchmarks: q = p + 2) on
        # ragged odd sizes with inflow data and a field over two coordinates
        dict(_transport("53x47x41", 3, 5, field="swirl", bc="inflow"), name="adv_53x47x41_p3q5_inflow"),
        # kinetic transport on a uniform 6D phase space (3 space, 3 velocity axes)
        dict(_transport("6x6x6x5x5x5", 2, 3, field="phase", bc="none"), name="adv6d_6_p2"),
        # learning a velocity field: forward and backward with beta per point
        {"name": "adjoint_48_p4", "kind": "adjoint", "mesh": "48x48x48", "p": 4, "q": 5, "bc": "periodic"},
        # SIPDG diffusion, GenDiL's Poisson rule q = p + 2, variable diffusivity
        {"name": "diffusion_64_p3q5", "kind": "diffusion", "mesh": "64x64x64", "p": 3, "q": 5, "basis": "gll",
         "mu": "trig", "bc": "periodic", "dtype": "f64"},
        # the same operator small, ragged, Legendre, Dirichlet boundaries, FP32
        {"name": "diffusion_27x23x19_p2q4_f32", "kind": "diffusion", "mesh": "27x23x19", "p": 2, "q": 4, "basis": "gl",
         "mu": "one", "bc": "dirichlet", "dtype": "f32"},
        # 6D phase space with per-element orders 1..3 (186 M unknowns)
        {"name": "padaptive6d_8_f32", "kind": "padaptive", "n": 8, "dtype": "f32"},
        # p-nonconforming domain decomposition: a p=1 block beside a p=3 block
        # (GenDiL's p-adaptivity test), cell terms and the interface between them
        {"name": "coupled_40_p1p3", "kind": "coupled", "mesh": "40x36x32", "p": 1, "p2": 3, "field": "c2"},
        # one implicit time step solved by restarted GMRES, FP32 inside FP64 refinement
        {"name": "gmres_mixed_32_p3", "kind": "solve", "n": 32, "p": 3, "method": "gmres_mixed"},
    ]


# (nodes, points) compiled for uniform transport operators, per dimension
_PAIRS = {2: [(2, 2), (3, 3), (3, 4), (4, 4), (4, 5)],
          3: [(2, 2), (2, 3), (2, 4), (3, 3), (3, 4), (3, 5), (4, 4), (4, 5), (4, 6), (5, 5), (5, 6), (5, 7), (6, 7)],
          4: [(2, 2), (2, 3), (3, 3), (3, 4), (4, 4), (4, 5)],
          6: [(2, 2), (2, 3), (3, 3)]}
_DIFF_PAIRS = {2: [(2, 3), (2, 4), (3, 4), (3, 5), (4, 4), (4, 5), (4, 6)],
               3: [(2, 3), (2, 4), (3, 3), (3, 4), (3, 5), (4, 4), (4, 5), (4, 6)]}
_TOP_DOFS = 16_777_216


def _sizes(rng, D, n, top=_TOP_DOFS, least=4, most=128):
    """Elements per axis: the total log-uniform from about least^D to `top` unknowns, the axes unequal."""
    lo, hi = D * math.log(least), min(math.log(top / n ** D), D * math.log(most))
    per = math.exp(rng.uniform(lo, max(lo, hi)) / D)
    while True:
        s = [max(1, round(per * math.exp(rng.uniform(-0.25, 0.25)))) for _ in range(D)]
        if math.prod(s) * n ** D <= top:
            return "x".join(str(v) for v in s)


def draw(rng):
    kind = rng.choices(["transport", "adjoint", "diffusion", "padaptive", "coupled", "faces", "solve"],
                       [9, 2, 4, 1, 2, 1, 1])[0]
    if kind == "transport":
        D = rng.choice([2, 3, 3, 3, 3, 4, 6])
        n, q = rng.choice(_PAIRS[D])
        fields = {2: ["rotating", "trig", "const", "swirl"], 3: ["c2", "rotating", "bubble", "swirl", "trig", "const"],
                  4: ["trig", "const", "phase"], 6: ["phase", "const", "phase"]}[D]
        op = rng.choice(["advection", "advection", "mass", "step"])
        return _transport(_sizes(rng, D, n, least=2 if D == 6 else 4, most=512 if D == 2 else 128), n - 1, q,
                          basis=rng.choice(["gll", "gll", "gl"]), field=rng.choice(fields),
                          bc="none" if op == "mass" else rng.choice(["periodic", "zero", "inflow", "none"]),
                          dtype=rng.choice(["f64", "f64", "f32"]), op=op, sigma=rng.choice(["one", "poly"]))
    if kind == "adjoint":
        n, q = rng.choice([(2, 2), (3, 3), (3, 4), (4, 4), (4, 5), (5, 5)])
        return {"kind": kind, "mesh": _sizes(rng, 3, n, 8_000_000), "p": n - 1, "q": q,
                "bc": rng.choice(["periodic", "zero"])}
    if kind == "diffusion":
        D = rng.choice([2, 3, 3, 3])
        n, q = rng.choice(_DIFF_PAIRS[D])
        return {"kind": kind, "mesh": _sizes(rng, D, n, 8_000_000, most=512 if D == 2 else 128), "p": n - 1, "q": q,
                "basis": rng.choice(["gll", "gl"]), "mu": rng.choice(["one", "trig"]),
                "bc": rng.choice(["periodic", "dirichlet"]), "dtype": rng.choice(["f64", "f64", "f32"])}
    if kind == "padaptive":
        return {"kind": kind, "n": rng.randint(3, 7), "dtype": rng.choice(["f32", "f64"])}
    if kind == "coupled":
        p, p2 = rng.choice([(1, 2), (2, 1), (1, 3), (3, 1), (2, 3), (3, 2), (2, 2)])
        return {"kind": kind, "mesh": _sizes(rng, 3, 4, 8_000_000), "p": p, "p2": p2,
                "field": rng.choice(["c2", "const", "rotating"])}
    if kind == "faces":
        n, q = rng.choice([(2, 2), (2, 3), (3, 3), (3, 4), (4, 4), (4, 5)])
        return {"kind": kind, "mesh": _sizes(rng, 3, n, 8_000_000), "p": n - 1, "q": q, "basis": "gll",
                "field": rng.choice(["c2", "rotating", "const"])}
    return {"kind": "solve", "n": rng.randint(6, 28), "p": rng.choice([1, 2, 3]),
            "method": rng.choice(["gmres", "gmres_mixed", "cg", "cg_mixed"])}


# ---------------------------------------------------------------------------
# the program's side: spaces, operators and inputs, then one pass
# ---------------------------------------------------------------------------

def _mesh_sizes(case):
    return [int(v) for v in case["mesh"].split("x")]


def _dtype(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.float64


def _fe(case, p):
    return (G.MakeLegendreFiniteElement if case.get("basis") == "gl" else G.MakeLobattoFiniteElement)(p)


def _periodic(case, D):
    if case.get("field") == "phase" and case["kind"] == "transport":  # space axes wrap, velocity axes do not
        return [d < D // 2 for d in range(D)]
    return [case.get("bc") == "periodic"] * D


def _space(case):
    M = _mesh_sizes(case)
    mesh = G.CartesianMesh(M, [1.0 / m for m in M], [0.0] * len(M), _periodic(case, len(M)))
    return G.MakeFiniteElementSpace(mesh, _fe(case, case["p"]))


def _random(shape, gen, dtype=torch.float64):
    return torch.rand(shape, generator=gen, device=DEVICE, dtype=dtype) * 2.0 - 1.0


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


STEP = 0.02  # adv_coef of the "step" operator and of the solves, times h below


def _bc(case):
    return {"zero": 0.0, "inflow": _field(BC_INFLOW_TERMS)}.get(case.get("bc"))


def _pointwise_shapes(M, q, periodic):
    D, E = len(M), math.prod(M)
    faces = [E // M[a] * (M[a] + (0 if periodic[a] else 1)) for a in range(D)]
    return (E, D, q ** D), [(f, q ** (D - 1)) for f in faces]


def _pointwise_field(case, gen):
    """beta at every cell point and its normal component at every face point: a
    mean flow plus 0.1 N(0, 1), as a field being fitted has."""
    M = _mesh_sizes(case)
    cell_shape, face_shapes = _pointwise_shapes(M, case["q"], _periodic(case, 3))
    mean = torch.tensor([1.0, 0.5, 0.25], dtype=torch.float64, device=DEVICE)
    cell = mean[None, :, None] + 0.3 * torch.randn(cell_shape, generator=gen, device=DEVICE, dtype=torch.float64)
    faces = [mean[a] + 0.3 * torch.randn(s, generator=gen, device=DEVICE, dtype=torch.float64)
             for a, s in enumerate(face_shapes)]
    return cell, faces


def _padaptive_orders(n):
    # one order map per mesh size: orders follow the solution, not the input
    return np.random.default_rng(2024 + n).choice(np.array([1, 2, 3], dtype=np.int8), size=n ** 6, p=[0.5, 0.35, 0.15])


def _solve_rhs_input(case, seed):
    """u0 at the nodes: a smooth bump plus small noise, M = n^3 elements of GLL order p."""
    n, N = case["n"], case["p"] + 1
    x1 = (torch.arange(n, dtype=torch.float64, device=DEVICE)[:, None] + torch.tensor(_rule_gll(N)[0], device=DEVICE)) / n
    g = torch.exp(-((x1 - 0.5) ** 2) / 0.02)  # [element, node]
    u = g[:, None, None, :, None, None] * g[None, :, None, None, :, None] * g[None, None, :, None, None, :]
    return u.reshape(-1).contiguous() + 1e-3 * _random(u.numel(), _gen(seed))


def prepare(case, seed):
    kind, gen = case["kind"], _gen(seed)
    if kind == "transport":
        fes, ir = _space(case), G.MakeIntegrationRule(case["q"])
        D = fes.dim
        sigma = _field(_sigma_terms(case["sigma"], D))
        beta = G.VectorField([_field(t) for t in _beta_terms(case["field"], D)])
        if case["op"] == "mass":
            op = G.MakeMassFiniteElementOperator(fes, ir, sigma)
        elif case["op"] == "advection":
            op = G.MakeAdvectionOperator(fes, ir, beta, _bc(case))
        else:
            op = G.MakeMassAdvectionOperator(fes, ir, beta, sigma, _bc(case), 1.0, STEP / max(fes.mesh.sizes))
        x = _random(op.num_dofs, gen, _dtype(case))
        return {"case": case, "op": op, "x": x, "y": torch.empty_like(x)}
    if kind == "adjoint":
        fes, ir = _space(case), G.MakeIntegrationRule(case["q"])
        cell, faces = _pointwise_field(case, gen)
        op = G.MakeAdvectionOperator(fes, ir, G.PointwiseField(cell, faces), _bc(case))
        u, gy = _random(op.num_dofs, gen), _random(op.num_dofs, gen)
        for t in (u, cell, *faces):
            t.requires_grad_(True)
        return {"case": case, "op": op, "u": u, "gy": gy, "cell": cell, "faces": faces}
    if kind == "diffusion":
        fes, ir = _space(case), G.MakeIntegrationRule(case["q"])
        op = G.MakeDiffusionOperator(fes, ir, _field(_mu_terms(case["mu"], fes.dim)), -1.0, float((case["p"] + 1) ** 2))
        x = _random(op.num_dofs, gen, _dtype(case))
        return {"case": case, "op": op, "x": x, "y": torch.empty_like(x)}
    if kind == "padaptive":
        n = case["n"]
        orders = _padaptive_orders(n)
        mesh = G.CartesianMesh([n] * 6, [1.0 / n] * 6, [0.0] * 6, [True, True, True, False, False, False])
        A = np.zeros((6, 6))
        A[0, 3] = A[1, 4] = A[2, 5] = 1.0
        op = G.MakeAdvectionOperator(G.MakePAdaptiveSpace(mesh, orders, orders + 1), None,
                                     G.AffineField(A, np.array([0.0, 0.0, 0.0, 0.1, 0.0, 0.0])))
        x = _random(op.num_dofs, gen, _dtype(case))
        return {"case": case, "op": op, "x": x, "y": torch.empty_like(x)}
    if kind == "coupled":
        M, p, p2 = _mesh_sizes(case), case["p"], case["p2"]
        h = [1.0 / m for m in M]
        fm = G.MakeFiniteElementSpace(G.CartesianMesh(M, h, [0.0] * 3), G.MakeLobattoFiniteElement(p))
        fp = G.MakeFiniteElementSpace(G.CartesianMesh(M, h, [1.0, 0.0, 0.0]), G.MakeLobattoFiniteElement(p2),
                                      G.L2Restriction(fm.num_dofs))
        beta = G.VectorField([_field(t) for t in _beta_terms(case["field"], 3)])
        ops = [G.MakeAdvectionOperator(f, G.MakeIntegrationRule(k + 1), beta) for f, k in ((fm, p), (fp, p2))]
        ops.append(G.MakeAdvectionFaceOperator(fm, fp, G.CartesianIntermeshFaceConnectivity(3, 3, M, M),
                                               G.MakeIntegrationRule(max(p, p2) + 2), beta))
        x = _random(fm.num_dofs + fp.num_dofs, gen)
        return {"case": case, "ops": ops, "x": x, "y": torch.empty_like(x)}
    if kind == "faces":
        fes = _space(case)
        op = G.MakeAdvectionFaceOperator(fes, G.MakeCartesianInteriorFaceConnectivity(fes.mesh.sizes),
                                         G.MakeIntegrationRule(case["q"]),
                                         G.VectorField([_field(t) for t in _beta_terms(case["field"], 3)]))
        x = _random(op.num_dofs, gen)
        return {"case": case, "op": op, "x": x, "y": torch.empty_like(x)}
    n, p = case["n"], case["p"]  # solve: (M + dt A) x = M u0, or M x = M u0
    fes = G.MakeFiniteElementSpace(G.CartesianMesh.unit(3, n), G.MakeLobattoFiniteElement(p))
    ir = G.MakeIntegrationRule(p + 1)
    mass = G.MakeMassFiniteElementOperator(fes, ir)
    if case["method"].startswith("cg"):
        K = mass
    else:
        K = G.MakeMassAdvectionOperator(fes, ir, G.VectorField([_field(t) for t in _beta_terms("c2", 3)]), bc=0.0,
                                        mass_coef=1.0, adv_coef=_solve_dt(n))
    b = torch.empty(K.num_dofs, dtype=torch.float64, device=DEVICE)
    mass(_solve_rhs_input(case, seed), b)
    return {"case": case, "op": K, "b": b, "x": torch.empty_like(b)}


def _solve_dt(n):
    return 0.5 / n / math.sqrt(3.5)  # half a cell per step at the field's largest speed


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("transport", "diffusion", "padaptive"):
        return state["op"](state["x"], state["y"])
    if kind == "adjoint":
        y = G.advection_apply(state["op"], state["u"], state["cell"], state["faces"])
        return (y.detach(), *torch.autograd.grad(y, [state["u"], state["cell"], *state["faces"]], state["gy"]))
    if kind == "coupled":
        for op in state["ops"]:  # the blocks overwrite their parts of y, the interface adds to both
            op(state["x"], state["y"])
        return state["y"]
    if kind == "faces":
        return state["op"](state["x"], state["y"].zero_())
    x = state["x"].zero_()
    getattr(G, case["method"])(state["op"], state["b"], x, rel_tol=1e-10)
    return x


# ---------------------------------------------------------------------------
# compulsory work and tolerances
# ---------------------------------------------------------------------------

def _sweeps(n, q, D, per=1):
    """Flops of one element's D one-dimensional contractions n -> q and back, `per` times."""
    return per * 2 * sum(2.0 * n ** (D - k) * q ** (k + 1) for k in range(D))


def work(case):
    kind = case["kind"]
    w = 4.0 if case.get("dtype") == "f32" else 8.0
    if kind in ("transport", "diffusion", "faces"):
        M = _mesh_sizes(case)
        D, n, q, E = len(M), case["p"] + 1, case["q"], math.prod(M)
        if kind == "diffusion":
            f = 2.0 * _sweeps(n, q, D)
        elif kind == "faces":
            f = 2.0 * D * _sweeps(n, q, D - 1)
        else:
            f = _sweeps(n, q, D) * (1.0 if case["op"] == "mass" else 1.5)
        return {"bytes": (2 if kind != "faces" else 3) * w * E * n ** D, "flops": E * f}
    if kind == "adjoint":
        M, n, q = _mesh_sizes(case), case["p"] + 1, case["q"]
        cs, fs = _pointwise_shapes(M, q, _periodic(case, 3))
        field = math.prod(cs) + sum(math.prod(s) for s in fs)
        E = math.prod(M)
        # u, gy and beta read; y, du and dbeta written
        return {"bytes": 8.0 * (4 * E * n ** 3 + 2 * field), "flops": 4.5 * E * _sweeps(n, q, 3)}
    if kind == "padaptive":
        n1 = _padaptive_orders(case["n"]).astype(np.float64) + 1
        # per unknown and axis one contraction with an n-column matrix on each side
        return {"bytes": 2 * w * float((n1 ** 6).sum()), "flops": float((2 * 2 * 6 * n1 ** 7).sum())}
    if kind == "coupled":
        E = math.prod(_mesh_sizes(case))
        ns = [case["p"] + 1, case["p2"] + 1]
        return {"bytes": 16.0 * E * sum(n ** 3 for n in ns), "flops": 1.5 * E * sum(_sweeps(n, n, 3) for n in ns)}
    # solve: nominal Krylov steps of the unpreconditioned system, each a pass over two vectors; the count
    # grows with the order only (the mass matrix's conditioning)
    N, n = (case["n"] * (case["p"] + 1)) ** 3, case["p"] + 1
    steps = {1: 60, 2: 200, 3: 600}[case["p"]]
    return {"bytes": 16.0 * N * steps, "flops": steps * case["n"] ** 3 * _sweeps(n, n, 3)}


def tolerance(case):
    """About four times what separates the start from exact() on the listed and drawn cases: 7e-8 for the solves
    (a relative residual of 1e-10 times the system's conditioning), 3e-7 in FP32, and in FP64 3e-15 and up to
    1e-14 for the Legendre bases of the highest orders."""
    if case["kind"] == "solve":
        return {"rel": 3e-7, "max": 1e-5}
    if case.get("dtype") == "f32":
        return {"rel": 1e-6, "max": 4e-5}
    return {"rel": 5e-14, "max": 2e-12}


# ---------------------------------------------------------------------------
# the same results in 64 bits from plain torch
# ---------------------------------------------------------------------------

def _rule_gl(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x + 1.0), 0.5 * w


def _rule_gll(n):
    """Gauss-Lobatto nodes and weights on [0, 1], n >= 2: the ends and the roots of P'_{n-1}."""
    P = np.polynomial.legendre.Legendre.basis(n - 1)
    d, dd = P.deriv(), P.deriv(2)
    inner = np.sort(np.real(d.roots())) if n > 2 else np.zeros(0)
    for _ in range(3):
        inner = inner - d(inner) / dd(inner)
    x = np.concatenate([[-1.0], inner, [1.0]])
    return 0.5 * (x + 1.0), 1.0 / (n * (n - 1) * P(x) ** 2)


def _lagrange(nodes, x):
    """Values and derivatives [len(x), len(nodes)] of the Lagrange basis on `nodes`."""
    n = len(nodes)
    V, dV = np.ones((len(x), n)), np.zeros((len(x), n))
    for i in range(n):
        others = [j for j in range(n) if j != i]
        for j in others:
            V[:, i] *= (x - nodes[j]) / (nodes[i] - nodes[j])
        for k in others:
            t = np.ones(len(x)) / (nodes[i] - nodes[k])
            for j in others:
                if j != k:
                    t *= (x - nodes[j]) / (nodes[i] - nodes[j])
            dV[:, i] += t
    return V, dV


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=DEVICE)


class _Basis:
    """1D tables of an n-node basis on the q-point Gauss rule."""

    def __init__(self, n, q, basis="gll"):
        nodes = (_rule_gl if basis == "gl" else _rule_gll)(n)[0]
        self.n, self.q = n, q
        xq, wq = _rule_gl(q)
        B, dB = _lagrange(nodes, xq)
        e, de = _lagrange(nodes, np.array([0.0, 1.0]))
        self.xq, self.w, self.B, self.dB = _t(xq), _t(wq), _t(B), _t(dB)
        self.end, self.dend = _t(e), _t(de)  # [end, node]


def _mul(mat, t, dim):
    """Contract dimension `dim` of t with the columns of mat."""
    return (t.movedim(dim, -1) @ mat.T).movedim(-1, dim)


class _Mesh:
    """A uniform space as a tensor [M_{D-1}, .., M_0, n, .., n]: axis a's
    elements are dimension D-1-a, its nodes or points dimension 2D-1-a."""

    def __init__(self, M, p, q, basis="gll", periodic=None, origin=None):
        self.M, self.D = list(M), len(M)
        self.b = _Basis(p + 1, q, basis)
        self.periodic = list(periodic) if periodic else [False] * self.D
        self.origin = list(origin) if origin else [0.0] * self.D
        self.h = [1.0 / m for m in M]
        self.detJ = math.prod(self.h)

    def ed(self, a):
        return self.D - 1 - a

    def pd(self, a):
        return 2 * self.D - 1 - a

    def shape(self, u):
        return u.double().reshape(self.M[::-1] + [self.b.n] * self.D)

    def coords(self, face=None, end=0):
        """Coordinates of the rule points, broadcastable; on axis `face` those of end 0 or 1."""
        X = []
        for a in range(self.D):
            xi = self.b.xq if a != face else _t([float(end)])
            e = torch.arange(self.M[a], dtype=torch.float64, device=DEVICE)
            x = self.origin[a] + self.h[a] * (e[:, None] + xi[None, :])
            s = [1] * (2 * self.D)
            s[self.ed(a)], s[self.pd(a)] = self.M[a], len(xi)
            X.append(x.reshape(s))
        return X

    def weights(self, face=None):
        W = 1.0
        for a in range(self.D):
            if a != face:
                s = [1] * (2 * self.D)
                s[self.pd(a)] = self.b.q
                W = W * self.b.w.reshape(s)
        return W

    def interp(self, u, skip=None):
        for a in range(self.D):
            if a != skip:
                u = _mul(self.b.B, u, self.pd(a))
        return u

    def test(self, v, skip=None):
        for a in range(self.D):
            if a != skip:
                v = _mul(self.b.B.T, v, self.pd(a))
        return v

    def across(self, t, a, end):
        """t of the neighbour across axis a's lower (0) or upper (1) face, and where there is one."""
        d, m = self.ed(a), self.M[a]
        s = [1] * (2 * self.D)
        s[d] = m
        inside = torch.ones(m, dtype=torch.bool, device=DEVICE)
        if not self.periodic[a]:
            inside[0 if end == 0 else m - 1] = False
        return torch.roll(t, 1 if end == 0 else -1, d), inside.reshape(s)


def _eval(terms, X):
    s = 0.0
    for scale, fns in terms:
        t = scale
        for a, f in fns.items():
            t = t * f(X[a])
        s = s + t
    return s


def _advection(m, u, cell_beta, face_beta, bc_terms=None, skip_boundary=True, cell=True):
    """A u for the shaped u: cell_beta(a) at the cell points, face_beta(a, end) at the face points."""
    b, y = m.b, 0.0
    if cell:
        uq = m.interp(u)
        for a in range(m.D):
            v = -(m.weights() * m.detJ / m.h[a]) * cell_beta(a) * uq
            for d in range(m.D):
                v = _mul(b.dB.T if d == a else b.B.T, v, m.pd(d))
            y = y + v
    for a in range(m.D):
        tr = [m.interp(_mul(b.end[e:e + 1], u, m.pd(a)), skip=a) for e in (0, 1)]
        for end in (0, 1):
            ext, inside = m.across(tr[1 - end], a, end)
            ext = torch.where(inside, ext, _outside(bc_terms, m, a, end))
            dot = face_beta(a, end) * ((1.0 if end else -1.0) / m.h[a])
            flux = m.weights(a) * m.detJ * dot * torch.where(dot > 0, tr[end], ext)
            if skip_boundary:
                flux = torch.where(inside, flux, torch.zeros((), dtype=torch.float64, device=DEVICE))
            y = y + _mul(b.end[end:end + 1].T, m.test(flux, skip=a), m.pd(a))
    return y


def _outside(bc_terms, m, a, end):
    g = _eval(bc_terms, m.coords(a, end)) if bc_terms else 0.0
    return g if isinstance(g, torch.Tensor) else torch.full((), float(g), dtype=torch.float64, device=DEVICE)


def _mass(m, u, sigma_terms):
    return m.test(m.weights() * m.detJ * _eval(sigma_terms, m.coords()) * m.interp(u))


def _separable_advection(m, u, terms, bc_terms=None, skip_boundary=True, cell=True):
    return _advection(m, u, lambda a: _eval(terms[a], m.coords()), lambda a, e: _eval(terms[a], m.coords(a, e)) + _t(0.0),
                      bc_terms, skip_boundary, cell)


def _diffusion(m, u, terms, sigma, kappa):
    """SIPDG with the reference's scaling: avg of mu grad u . n and jumps with the normal s e_a / h_a."""
    b, y, uq = m.b, 0.0, m.interp(u)
    c = m.weights() * m.detJ * _eval(terms, m.coords())
    for a in range(m.D):
        g = u
        for d in range(m.D):
            g = _mul(b.dB if d == a else b.B, g, m.pd(d))
        v = c * g / m.h[a] ** 2
        for d in range(m.D):
            v = _mul(b.dB.T if d == a else b.B.T, v, m.pd(d))
        y = y + v
    del uq, c
    for a in range(m.D):
        ih = 1.0 / m.h[a]
        val = [m.interp(_mul(b.end[e:e + 1], u, m.pd(a)), skip=a) for e in (0, 1)]
        der = [m.interp(_mul(b.dend[e:e + 1], u, m.pd(a)), skip=a) for e in (0, 1)]
        for end in (0, 1):
            mu = _eval(terms, m.coords(a, end))
            nv, inside = m.across(val[1 - end], a, end)
            ng, _ = m.across(der[1 - end], a, end)
            avg = mu * ih * torch.where(inside, 0.5 * (der[end] + ng), der[end])
            jump = torch.where(inside, val[end] - nv, val[end])
            half = torch.where(inside, 0.5, 1.0).double()
            n, w = (1.0 if end else -1.0) * ih, m.weights(a) * m.detJ
            du = -w * avg * n + w * kappa * ih * ih * mu * jump
            dg = sigma * w * jump * mu * half * n * ih
            y = y + _mul(b.end[end:end + 1].T, m.test(du, skip=a), m.pd(a))
            y = y + _mul(b.dend[end:end + 1].T, m.test(dg, skip=a), m.pd(a))
    return y


def _padaptive(case, x):
    """Advection by beta = (X3, X4, X5, 0.1, 0, 0), element batches by order, both
    sides of a face on the rule of max(n, n_neighbour) points."""
    n_el, D = case["n"], 6
    orders = torch.as_tensor(_padaptive_orders(n_el).astype(np.int64), device=DEVICE)
    nn, h = orders + 1, 1.0 / n_el
    off = torch.cumsum(nn ** D, 0) - nn ** D
    E = n_el ** D
    sub = [(torch.arange(E, device=DEVICE) // n_el ** a) % n_el for a in range(D)]
    x, y = x.double(), torch.zeros(x.numel(), dtype=torch.float64, device=DEVICE)
    bases = {(n, q): _Basis(n, q) for n in (2, 3, 4) for q in (2, 3, 4) if q >= n}

    def pd(a):
        return D - a  # [elements, n (axis 5), .., n (axis 0)]

    def beta(c, el, q, face=None, end=0):
        if c > 3:
            return None
        src = c + 3
        if c == 3:
            return torch.full([1] * (D + 1), 0.1, dtype=torch.float64, device=DEVICE)
        xi = bases[(2, q)].xq if src != face else _t([float(end)])
        s = [len(el)] + [1] * D
        s[pd(src)] = len(xi)
        return (h * (sub[src][el].double()[:, None] + xi[None, :])).reshape(s)

    def weights(q, face=None):
        W = 1.0
        for a in range(D):
            if a != face:
                s = [1] * (D + 1)
                s[pd(a)] = q
                W = W * bases[(2, q)].w.reshape(s)
        return W

    def gather(el, n):
        idx = off[el][:, None] + torch.arange(n ** D, device=DEVICE)[None, :]
        return x[idx].reshape([len(el)] + [n] * D)

    detJ = h ** D
    for n in (2, 3, 4):
        for el in torch.split(torch.nonzero(nn == n).reshape(-1), 2 ** 23 // n ** D * 2):
            b = bases[(n, n)]
            u = gather(el, n)
            uq = u
            for a in range(D):
                uq = _mul(b.B, uq, pd(a))
            out = 0.0
            for c in range(4):
                v = -(weights(n) * detJ / h) * beta(c, el, n) * uq
                for d in range(D):
                    v = _mul(b.dB.T if d == c else b.B.T, v, pd(d))
                out = out + v
            for c in range(4):  # beta >= 0: lower faces take the neighbour's trace, upper faces their own
                for end in (1, 0):
                    s_nb = sub[c][el] + (1 if end else -1)
                    has = (s_nb >= 0) & (s_nb < n_el) | (c < 3)  # the space axes wrap
                    nb = el + (s_nb % n_el - sub[c][el]) * n_el ** c
                    for k in (2, 3, 4):
                        pick = torch.nonzero(has & (nn[nb] == k)).reshape(-1)
                        if not len(pick):
                            continue
                        q = max(n, k)
                        bo, bn, e = bases[(n, q)], bases[(k, q)], el[pick]
                        if end == 1:
                            src, bs, row = u[pick], bo, bo.end[1:2]
                        else:
                            src, bs, row = gather(nb[pick], k), bn, bn.end[1:2]
                        t = _mul(row, src, pd(c))
                        for d in range(D):
                            if d != c:
                                t = _mul(bs.B, t, pd(d))
                        t = t * (weights(q, c) * detJ / h * (1.0 if end else -1.0)) * beta(c, e, q, c, end)
                        for d in range(D):
                            if d != c:
                                t = _mul(bo.B.T, t, pd(d))
                        out = out.index_add(0, pick, _mul(bo.end[end:end + 1].T, t, pd(c)))
            idx = off[el][:, None] + torch.arange(n ** D, device=DEVICE)[None, :]
            y[idx] = out.reshape(len(el), -1)
    return y


def _pointwise(m, t, q, a=None):
    """A per-point array [entities, q^k] as a tensor over (element or face grid, points)."""
    ext = [m.M[d] + (1 if d == a and not m.periodic[d] else 0) for d in range(m.D)]
    pts = [1 if d == a else q for d in range(m.D)]
    return t.reshape(ext[::-1] + pts[::-1])


def _exact_adjoint(case, seed):
    gen = _gen(seed)
    M, q = _mesh_sizes(case), case["q"]
    m = _Mesh(M, case["p"], q, periodic=_periodic(case, 3))
    cell, faces = _pointwise_field(case, gen)
    N = math.prod(M) * m.b.n ** 3
    u, gy = _random(N, gen), _random(N, gen)
    for t in (u, cell, *faces):
        t.requires_grad_(True)

    def face_beta(a, end):
        t = _pointwise(m, faces[a], q, a)
        if m.periodic[a]:
            return t if end == 0 else torch.roll(t, -1, m.ed(a))
        return t.narrow(m.ed(a), end, m.M[a])

    bc = [(0.0, {})] if case["bc"] == "zero" else None
    y = _advection(m, m.shape(u), lambda a: _pointwise(m, cell[:, a], q), face_beta, bc, bc is None).reshape(-1)
    return (y.detach(), *torch.autograd.grad(y, [u, cell, *faces], gy))


def _exact_solve(case, seed):
    """(M + dt A) x = M u0 by refinement with the exact inverse of M as the
    preconditioner of GMRES, to about 1e-14; M x = M u0 is u0."""
    u0 = _solve_rhs_input(case, seed)
    if case["method"].startswith("cg"):
        return u0
    n, N = case["n"], case["p"] + 1
    m = _Mesh([n] * 3, case["p"], N)
    M1 = m.b.B.T @ torch.diag(m.b.w) @ m.b.B
    inv = torch.linalg.inv(M1) * n
    terms, dt = _beta_terms("c2", 3), _solve_dt(n)

    def K(v):  # v + dt M^-1 A v
        a = _separable_advection(m, m.shape(v), terms, None, False)
        for d in range(3):
            a = _mul(inv, a, m.pd(d))
        return v + dt * a.reshape(-1)

    x = u0.clone()
    for _ in range(4):
        r = u0 - K(x)
        beta = r.norm()
        if beta <= 1e-15 * u0.norm():
            break
        V, H = [r / beta], torch.zeros(31, 30, dtype=torch.float64, device=DEVICE)
        for k in range(30):
            w = K(V[k])
            for _ in range(2):
                for i, v in enumerate(V):
                    c = v @ w
                    H[i, k] += c
                    w = w - c * v
            H[k + 1, k] = w.norm()
            V.append(w / H[k + 1, k])
        e = torch.zeros(31, 1, dtype=torch.float64, device=DEVICE)
        e[0] = beta
        z = torch.linalg.lstsq(H, e).solution.reshape(-1)
        x = x + sum(z[k] * V[k] for k in range(30))
    return x


def exact(case, seed):
    kind, gen = case["kind"], _gen(seed)
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    if kind == "solve":
        return _exact_solve(case, seed)
    if kind == "padaptive":
        N = int(((_padaptive_orders(case["n"]).astype(np.int64) + 1) ** 6).sum())
        return _padaptive(case, _random(N, gen, _dtype(case)))
    M = _mesh_sizes(case)
    D = len(M)
    if kind == "coupled":
        return _exact_coupled(case, gen)
    m = _Mesh(M, case["p"], case["q"], case["basis"], _periodic(case, D))
    x = _random(math.prod(M) * m.b.n ** D, gen, _dtype(case))
    u = m.shape(x)
    if kind == "diffusion":
        return _diffusion(m, u, _mu_terms(case["mu"], D), -1.0, float((case["p"] + 1) ** 2)).reshape(-1)
    if kind == "faces":
        return _separable_advection(m, u, _beta_terms(case["field"], 3), cell=False).reshape(-1)
    y = 0.0
    if case["op"] != "advection":
        y = y + _mass(m, u, _sigma_terms(case["sigma"], D))
    if case["op"] != "mass":
        bc = {"zero": [(0.0, {})], "inflow": BC_INFLOW_TERMS}.get(case["bc"])
        c = 1.0 if case["op"] == "advection" else float(np.float32(STEP / max(M)) if case["dtype"] == "f32" else STEP / max(M))
        y = y + c * _separable_advection(m, u, _beta_terms(case["field"], D), bc, bc is None)
    return y.reshape(-1)


def _exact_coupled(case, gen):
    M, ps = _mesh_sizes(case), (case["p"], case["p2"])
    terms, q = _beta_terms(case["field"], 3), max(ps) + 2
    sizes = [math.prod(M) * (p + 1) ** 3 for p in ps]
    x = _random(sum(sizes), gen)
    parts, y, traces, meshes = torch.split(x, sizes), [], [], []
    for i, p in enumerate(ps):
        m = _Mesh(M, p, p + 1, origin=[float(i), 0.0, 0.0])
        y.append(_separable_advection(m, m.shape(parts[i]), terms))
        f = _Mesh(M, p, q, origin=[float(i), 0.0, 0.0])  # the interface's shared rule
        t = f.interp(_mul(f.b.end[1 - i:2 - i], f.shape(parts[i]), f.pd(0)), skip=0)
        traces.append(t.narrow(f.ed(0), M[0] - 1 if i == 0 else 0, 1))
        meshes.append(f)
    f = meshes[0]
    beta = _eval(terms[0], [c.narrow(f.ed(0), M[0] - 1, 1) if a == 0 else c for a, c in enumerate(f.coords(0, 1))])
    dot = beta * (1.0 / f.h[0]) + _t(0.0)
    flux = f.weights(0) * f.detJ * dot * torch.where(dot > 0, traces[0], traces[1])
    for i, f in enumerate(meshes):
        v = _mul(f.b.end[1 - i:2 - i].T, f.test(flux, skip=0), f.pd(0)) * (1.0 if i == 0 else -1.0)
        y[i].narrow(f.ed(0), M[0] - 1 if i == 0 else 0, 1).add_(v)
    return torch.cat([t.reshape(-1) for t in y])
