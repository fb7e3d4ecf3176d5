"""Arnoldi steps whose passes sum each other's partials: every count of stored
vectors up to the largest, on one block, on a part of a block's sums, on the
largest grids (512 blocks up to 8 vectors, then 256) with a tail after the last
pack, and cycles that end early, against dense FP64 algebra."""
import numpy as np
import pytest
import torch

from gendil_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,m,stop", [(700, 32, 32), (70_003, 32, 32), (70_003, 32, 9), (4_300_007, 32, 32),
                                      (4_300_007, 9, 8), (70_003, 5, 1)])
def test_cycle_minimises_the_residual(n, m, stop, dtype):
    check_cycle(n, m, stop, dtype, n + (-n) % 4, 0)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,m,stop", [(700, 32, 32), (70_003, 32, 9), (70_003, 5, 1), (4_300_007, 32, 32)])
@pytest.mark.parametrize("offset", [0, 1])
def test_cycle_on_a_basis_that_no_16_bytes_align(n, m, stop, dtype, offset):
    """One value per access: an odd leading dimension, and V and x one element off."""
    check_cycle(n, m, stop, dtype, n + 1 - n % 2, offset)


def check_cycle(n, m, stop, dtype, ldv, offset):
    lib = L.lib()
    st = torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(n + m)
    d = 1.0 + torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    b = torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
    V = torch.zeros(offset + (m + 1) * ldv, dtype=dtype, device="cuda")[offset:].view(m + 1, ldv)
    ws = torch.randint(0, 255, (lib.gd_gmres_workspace_bytes(),), generator=g, dtype=torch.uint8, device="cuda")
    step = lib.gd_arnoldi_step_f64 if dtype == torch.float64 else lib.gd_arnoldi_step_f32
    upd = lib.gd_gmres_update_f64 if dtype == torch.float64 else lib.gd_gmres_update_f32
    x = torch.zeros(offset + n, dtype=torch.float64, device="cuda")[offset:]
    # the check's own sums of n products round like a walk of n steps, sqrt(n) eps
    # (4.6e-13 at the largest n: the first vector, normalised by torch, shows 6e-14)
    tol = max(1e-13, n**0.5 * 2.0**-52) if dtype == torch.float64 else 1e-6
    for _ in range(2):  # the second cycle starts on the first one's workspace
        V[0, :n] = (b / b.norm()).to(dtype)
        L.check(lib.gd_gmres_begin(ws.data_ptr(), float(b.norm()), 1.0, st), "begin")
        resid = torch.full((m,), -1.0, dtype=torch.float64, device="cuda")
        for k in range(stop):
            V[k + 1, :n] = (d * V[k, :n].double()).to(dtype)
            L.check(step(n, m, k, V.data_ptr(), ldv, ws.data_ptr(), resid[k:].data_ptr(), st), "step")
        x.zero_()
        L.check(upd(n, m, stop, V.data_ptr(), ldv, ws.data_ptr(), x.data_ptr(), st), "update")
        Q = V[: stop + 1, :n].double()
        gram = Q @ Q.T
        assert float((gram - torch.eye(stop + 1, dtype=torch.float64, device="cuda")).abs().max()) <= tol
        # every residual estimate against the least-squares residual over the same space
        KQ = d * Q[:stop]
        G, rhs = (KQ @ KQ.T).cpu().numpy(), (KQ @ b).cpu().numpy()
        r = resid.cpu().numpy()
        assert np.all(r[:stop] > 0) and np.all(r[stop:] == -1.0)
        for k in (0, stop // 2, stop - 1):
            y = np.linalg.solve(G[: k + 1, : k + 1], rhs[: k + 1])
            true = float((b - torch.as_tensor(y, device="cuda") @ KQ[: k + 1]).norm())
            assert abs(r[k] - true) <= (1e-10 if dtype == torch.float64 else 1e-5) * float(b.norm())
        assert abs(float((b - d * x).norm()) - r[stop - 1]) <= (1e-10 if dtype == torch.float64 else 1e-5) * float(b.norm())
