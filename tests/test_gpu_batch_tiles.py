"""The batched mixed solve spread over tiles (reduced CG, several workgroups a
system) against the FP64 batch solve: systems of one row pair to many tiles,
5- and 7-point rows, sizes around a tile's, and a system whose tiles' sums
need more than one round of words; batches of small systems only, which keep
one workgroup a system.  Every system's solution meets the true
residual test, checked on the host with the oracle's product; repeated solves
are equal bit for bit (every sum has a fixed order)."""
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


@pytest.fixture(scope="module")
def pp(torch):
    import prispack_amd
    return prispack_amd


def vardiff(side, seed):
    return ppo.vardiff2d(side, np.exp(ppo.normal(side * side, seed)))


BATCHES = {
    "small": lambda: [ppo.laplacian(2, 1, 1), ppo.laplacian(3, 2, 1), vardiff(5, 1), vardiff(16, 2)],  # one workgroup
    "small_beside_a_larger": lambda: [ppo.laplacian(2, 1, 1), ppo.laplacian(3, 2, 1), vardiff(5, 1), vardiff(16, 2),
                                      vardiff(25, 3)],
    "below_the_line": lambda: [ppo.laplacian(599, 1, 1), ppo.laplacian(23, 26, 1)],
    "at_the_line": lambda: [ppo.laplacian(600, 1, 1), ppo.laplacian(23, 26, 1)],
    "below_the_line_3d": lambda: [ppo.laplacian(7, 157, 1), ppo.laplacian(10, 11, 9)],  # 1099 rows and less
    "at_the_line_3d": lambda: [ppo.laplacian(10, 11, 10), ppo.laplacian(5, 4, 3)],
    "around_a_tile": lambda: [vardiff(s, s) for s in (45, 46, 63, 64, 65, 90, 91)],
    "around_a_slice": lambda: [ppo.laplacian(*g, 1) for g in ((17, 15), (16, 16), (257, 1), (73, 7), (32, 16), (2, 1),
                                                              (31, 20))],
    "uneven": lambda: [vardiff(s, s) for s in (200, 33, 129, 8, 70)],
    "seven_point": lambda: [ppo.laplacian(16, 15, 14), ppo.laplacian(24, 23, 22), vardiff(40, 3)],
    "many_tiles": lambda: [ppo.laplacian(90, 2100, 1), vardiff(20, 5)],
    "halo_too_wide": lambda: [vardiff(400, 4), vardiff(20, 5)],  # stays with one workgroup a system
}


@pytest.mark.parametrize("name", list(BATCHES))
def test_tiled_mixed_solve(pp, torch, name):
    systems = BATCHES[name]()
    B = pp.BatchedSystems(systems, ordering=1)
    xt = np.concatenate([ppo.normal(len(A[0]) - 1, 60 + s) for s, A in enumerate(systems)])
    b = torch.tensor(np.concatenate([ppo.spmv(A, xt[B.row_off[s]:B.row_off[s + 1]]) for s, A in enumerate(systems)]),
                     device="cuda")
    print(f"[tiles] {name} n={B.n}", flush=True)
    x64, x, y = (torch.zeros_like(b) for _ in range(3))
    it64 = B.solve(b, x64, precision="fp64", tol=1e-8)
    it = B.solve(b, x, precision="mixed", tol=1e-8)
    assert B.report.converged and B.report.true_relres < 1e-8 and B.report.cg_variant == 3
    # the path under test ran: every system a tile at least
    if name in ("halo_too_wide", "small", "below_the_line", "below_the_line_3d"):
        assert B.info().tiles == B.report.batch_tiles == 0
    else:
        assert B.info().tiles == B.report.batch_tiles >= len(systems)
    assert np.array_equal(it, B.solve(b, y, precision="mixed", tol=1e-8)) and torch.equal(x, y)
    for s in range(len(systems)):
        lo, hi = int(B.row_off[s]), int(B.row_off[s + 1])
        u, v, bs = (t[lo:hi].cpu().numpy() for t in (x, x64, b))
        # the solve's own test, ||b - A x|| <= 1e-8 ||b||, with the rounding of
        # two FP64 residuals (1e-16 of ||A|| ||x||, far below a hundredth of it) on top
        assert np.linalg.norm(bs - ppo.spmv(systems[s], u)) <= 1.01e-8 * np.linalg.norm(bs), s
        # so A (u - v) is at most the two residuals together; FlexibleCG stops
        # on its recursive residual, within a tenth of the true one here
        assert np.linalg.norm(ppo.spmv(systems[s], u - v)) <= 2.2e-8 * np.linalg.norm(bs), s
        # an FP32 restart costs some iterations over the FP64 solve's
        assert it[s] <= 1.3 * it64[s] + 20, (s, it[s], it64[s])


def test_tiled_solve_stops_at_its_iteration_limit(pp, torch):
    B = pp.BatchedSystems([vardiff(150, 1), vardiff(30, 2)], ordering=1)
    b = torch.ones(B.n, dtype=torch.float64, device="cuda")
    x = torch.zeros_like(b)
    it = B.solve(b, x, precision="mixed", tol=1e-8, maxit=25)
    assert not B.report.converged and it.max() <= 25 and B.report.batch_tiles > 0
    # a zero right-hand side needs no iteration
    b[:B.row_off[1]] = 0.0
    it = B.solve(b, x, precision="mixed", tol=1e-8)
    assert it[0] == 0 and B.report.converged and bool((x[:int(B.row_off[1])] == 0).all())
