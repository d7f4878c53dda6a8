"""GMRES's orthogonalisation passes and step kernel: the residual estimates of
the first cycle against the oracle's, for row counts around one workgroup
(256, 1024 rows) and around all of the grid (four workgroups of 256 per CU),
column counts over every register slot up to 32 and past them, with and
without a preconditioner and with either variant; the FP32 basis to its
converged residual."""
import numpy as np
import pytest

from oracle import ppo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


GRIDS = [(2, 1, 1), (17, 15, 1), (16, 16, 1), (257, 1, 1), (41, 25, 1), (65, 63, 65)]


@pytest.mark.parametrize("flexible", [1, 0])
@pytest.mark.parametrize("restart", [3, 31, 45])
@pytest.mark.parametrize("grid", GRIDS)
def test_first_cycle_against_oracle(torch, grid, restart, flexible):
    import prispack_amd as pp
    # diagonal shifted by 0.05: eigenvalues in [0.05, 12.05]
    A = ppo.laplacian(*grid, shift=-0.05)
    n = len(A[0]) - 1
    b = ppo.normal(n, 4)
    steps = min(restart, n - 1)
    want = np.asarray(ppo.gmres(A, b, None, tol=1e-13, restart=restart, flexible=bool(flexible))["hist"])
    M = pp.CSRMatrix(*A)
    S = pp.GMRES(n, None, tolerance=1e-13, GMRESType=pp.FlexibleGMRES if flexible else pp.NormalGMRES)
    S.setRestart(True, restart)
    S.opts.record_history = 1
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    S.solve(M, torch.tensor(b, device="cuda"), x)
    got = S.history()
    k = min(len(got), len(want), steps)
    assert k >= 1
    # rounding of the basis, amplified by at most the condition number, a step
    tol = 64 * 2.0 ** -52 * 241 * steps
    np.testing.assert_allclose(got[:k], want[:k], rtol=0, atol=tol)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("grid", GRIDS)
def test_preconditioned_residual(torch, grid, precision):
    import prispack_amd as pp
    A = ppo.upwind(*grid, 5.0, 2.0, 1.0)
    n = len(A[0]) - 1
    b = ppo.normal(n, 5)
    M = pp.CSRMatrix(*A)
    P = pp.ILU0(M, make_f32=precision == "mixed")
    S = pp.GMRES(n, P, tolerance=1e-9, precision=precision)
    S.setRestart(True, 30)
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    S.solve(M, torch.tensor(b, device="cuda"), x)
    assert S.getConvergence()
    r = b - ppo.spmv(A, x.cpu().numpy())
    # the estimate is below 1e-9; the residual itself adds the basis's
    # rounding, 2^-24 of the cycle's first residual in FP32
    assert np.linalg.norm(r) <= 1.1e-9 * np.linalg.norm(b) * (1 if precision == "fp64" else 10)


@pytest.mark.parametrize("launch", [0, 1])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [3, 1025, 700_001])
def test_stop_inside_a_cycle(torch, n, precision, launch):
    # three distinct eigenvalues: the third step of every cycle stops it, on
    # one workgroup and on all of the grid, the same bits each time
    import prispack_amd as pp
    d = np.array([1.0, 2.0, 5.0])[np.arange(n) % 3]
    M = pp.CSRMatrix(np.arange(n + 1, dtype=np.uint32), np.arange(n, dtype=np.uint32), d)
    b = torch.tensor(ppo.normal(n, 6), device="cuda")
    out = []
    for _ in range(3):
        S = pp.GMRES(n, None, tolerance=1e-9, precision=precision)
        S.setRestart(True, 30)
        S.opts.launch = launch
        x = torch.zeros_like(b)
        S.solve(M, b, x)
        assert S.getConvergence()
        r = b - torch.tensor(d, device="cuda") * x
        assert float(r.norm()) <= 1.1e-9 * float(b.norm()) * (1 if precision == "fp64" else 10)
        out.append((S.getNumIter(), x))
    for it, x in out[1:]:
        assert it == out[0][0] and torch.equal(x, out[0][1])
