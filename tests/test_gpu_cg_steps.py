"""FlexibleCG's vector updates, which add up the partial sums of the kernels
before them: the residual history of every check against the oracle's, for
row counts around one workgroup (1024 rows) and around all of the grid (two
workgroups per CU), with the first forward level taken along (colour-ordered
IC(0)) and without, in FP64."""
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


def parity_order(nx, ny, nz):
    """Row order of the two-colour ordering: even points first, each in grid order."""
    i = np.arange(nx * ny * nz)
    return np.argsort((i % nx + i // nx % ny + i // (nx * ny)) % 2, kind="stable")


def permute(A, order):
    n = len(order)
    rp, ci, v = A
    new = np.empty(n, np.int64)
    new[order] = np.arange(n)
    rows = np.repeat(np.arange(n), np.diff(rp.astype(np.int64)))
    r2, c2 = new[rows], new[ci]
    at = np.lexsort((c2, r2))
    return (np.concatenate([[0], np.cumsum(np.bincount(r2, minlength=n))]).astype(np.uint32),
            c2[at].astype(np.uint32), v[at])


@pytest.mark.parametrize("precond", ["ic0_coloured", "ic0", "none"])
@pytest.mark.parametrize("grid", [(1, 1, 1), (2, 1, 1), (33, 31, 1), (32, 32, 1), (41, 25, 1), (89, 71, 83)])
def test_history_against_oracle(torch, grid, precond):
    import prispack_amd as pp
    # diagonal shifted by one: eigenvalues in [1, 13], so the recurrences
    # differ from the oracle's by rounding only, a few eps x 13 per iteration
    A = ppo.laplacian(*grid, shift=-1.0)
    n = len(A[0]) - 1
    b = ppo.normal(n, 3)
    order = parity_order(*grid) if precond == "ic0_coloured" else np.arange(n)
    Ao = permute(A, order)
    want = ppo.cg(Ao, b[order], None if precond == "none" else ppo.Prec(Ao, "ic0"), tol=1e-10, maxit=100)
    M = pp.CSRMatrix(*A)
    P = None
    if precond != "none":
        P = pp.IC0(M, ordering=int(precond == "ic0_coloured"))
        P.setup()
    S = pp.CG(n, P, tol=1e-10, maxIter=100).setCGVariant("reference")
    S.opts.record_history = 1
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    S.solve(M, torch.tensor(b, device="cuda"), x)
    xo = np.empty(n)
    xo[order] = want["x"]
    eps = 64 * 2.0 ** -52 * 13 * max(1, want["iters"])
    assert S.getConvergence() == want["converged"]
    assert abs(S.getNumIter() - want["iters"]) <= 1
    got = x.cpu().numpy()
    # both stop below 1e-10: that and the rounding bound the difference
    assert np.linalg.norm(got - xo) <= (2e-10 + eps) * np.linalg.norm(b)
    h, ho = S.history(), np.asarray(want["hist"])
    k = min(len(h), len(ho))
    assert k >= min(want["iters"], 1)
    np.testing.assert_allclose(h[:k], ho[:k], rtol=0, atol=eps)


def _blocks2(count, block):
    """count copies of a 2 x 2 block on the diagonal."""
    n = 2 * count
    cols = np.repeat(np.arange(n) // 2 * 2, 2) + np.tile([0, 1], n)
    return np.arange(0, 2 * n + 1, 2, dtype=np.uint32), cols.astype(np.uint32), np.tile(np.ravel(block), count)


# [[1, 1], [1, 1]] with b = (1, 0): step 1 goes to x = (1, 0), step 2 has (d, A d) = 0;
# [[0, 1], [1, 0]] with b = (1, 0): (d, A d) = 0 at once; all of it in small whole numbers
@pytest.mark.parametrize("launch", [0, 1])
@pytest.mark.parametrize("count", [1, 513, 350_001])
@pytest.mark.parametrize("block,x", [([[1, 1], [1, 1]], (1.0, 0.0)), ([[0, 1], [1, 0]], (0.0, 0.0)),
                                     ([[1, np.nan], [np.nan, 1]], (0.0, 0.0))])
def test_breakdown_leaves_x_at_the_step_before(torch, block, x, count, launch):
    import prispack_amd as pp
    M = pp.CSRMatrix(*_blocks2(count, np.array(block, float)))
    b = np.tile([1.0, 0.0], count)
    for host in (False, True):
        S = pp.CG(M.n, None, tol=1e-10, maxIter=50).setCGVariant("reference")
        S.opts.launch = launch
        got = np.zeros(M.n) if host else torch.zeros(M.n, dtype=torch.float64, device="cuda")
        with pytest.raises(pp.PrisPackError) as e:
            S.solve(M, b if host else torch.tensor(b, device="cuda"), got)
        assert e.value.status == (8 if np.isnan(block).any() else 7) and not S.getConvergence()
        assert np.array_equal(got if host else got.cpu().numpy(), np.tile(x, count))
