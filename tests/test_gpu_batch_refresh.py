"""New values of a batch factored on the device (pp_batch_set_values) against
a batch set up from scratch on them: the same factor and operators bit for
bit, hence the same solves, in both orderings and precisions, from host and
device arrays, for sizes around the workgroup's and a one-row system; pivots
that fail and patterns outside the device path behave as the host's."""
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


def scaled(systems, seed):
    """D A D of every system: same pattern, still SPD."""
    out = []
    for s, (rp, ci, v) in enumerate(systems):
        n = len(rp) - 1
        d = np.exp(0.4 * ppo.normal(n, seed + s))
        rows = np.repeat(np.arange(n), np.diff(rp.astype(np.int64)))
        out.append((rp, ci, d[rows] * v * d[ci]))
    return out


def solves(torch, B, b):
    out = []
    for precision in ("fp64", "mixed"):
        x = torch.zeros_like(b)
        its = B.solve(b, x, precision=precision, tol=1e-8)
        assert B.report.converged
        out.append((its.copy(), x))
    return out


@pytest.mark.parametrize("on_device", [False, True])
@pytest.mark.parametrize("ordering", [0, 1])
def test_refresh_matches_fresh_batch(pp, torch, ordering, on_device):
    sides = [2, 7, 31, 32, 33, 45]  # 33^2 rows: one past the workgroup's
    systems = [ppo.vardiff2d(s, np.exp(ppo.normal(s * s, 40 + s))) for s in sides]
    if ordering == 0:
        systems.append((np.array([0, 1], np.uint32), np.array([0], np.uint32), np.array([2.5])))
        systems.append(ppo.laplacian(9, 8, 7))
    B = pp.BatchedSystems(systems, ordering=ordering)
    b = torch.tensor(np.concatenate([ppo.uniform(len(A[0]) - 1, 5 + s) for s, A in enumerate(systems)]), device="cuda")
    for step in range(2):
        new = scaled(systems, 100 * (step + 1))
        v = np.concatenate([A[2] for A in new])
        B.set_values(torch.tensor(v, device="cuda") if on_device else v)
        assert B.info().device_refactors == step + 1  # not the host's factorization
        F = pp.BatchedSystems(new, ordering=ordering)
        for (i0, x0), (i1, x1) in zip(solves(torch, B, b), solves(torch, F, b)):
            assert np.array_equal(i0, i1) and torch.equal(x0, x1)
    # another order after values set on the device
    B.set_ordering(1 - ordering)
    F.set_ordering(1 - ordering)
    if ordering == 1:
        for (i0, x0), (i1, x1) in zip(solves(torch, B, b), solves(torch, F, b)):
            assert np.array_equal(i0, i1) and torch.equal(x0, x1)


@pytest.mark.parametrize("ordering", [0, 1])
def test_failing_pivot_keeps_the_factor_in_use(pp, torch, ordering):
    # as after a failed factorization on the host: the new values, the factor of
    # the ones before.  Three FP64 iterations against the oracle's with just that.
    from mc_order import greedy_order, permute
    from prispack_amd import PrisPackError
    systems = [ppo.vardiff2d(s, np.exp(ppo.normal(s * s, 40 + s))) for s in (9, 33, 12)]
    B = pp.BatchedSystems(systems, ordering=ordering)
    b = torch.tensor(np.concatenate([ppo.uniform(len(A[0]) - 1, 5 + s) for s, A in enumerate(systems)]), device="cuda")
    for step in range(2):
        good = scaled(systems, 700) if step else systems
        if step:
            B.set_values(np.concatenate([A[2] for A in good]))
        for fail in range(2):  # twice: the factor stays that of the good values
            bad = scaled(systems, 800 + fail)
            rp, ci, v = bad[1]
            v[np.flatnonzero((ci == 77) & (np.repeat(np.arange(len(rp) - 1), np.diff(rp.astype(int))) == 77))] *= -1.0
            with pytest.raises(PrisPackError) as e:
                B.set_values(torch.tensor(np.concatenate([A[2] for A in bad]), device="cuda"))
            assert e.value.status == 3 and "system 1" in str(e.value)
            x = torch.zeros_like(b)
            B.solve(b, x, precision="fp64", tol=1e-300, maxit=3)
            for s in range(len(systems)):
                lo, hi = int(B.row_off[s]), int(B.row_off[s + 1])
                order = greedy_order(systems[s])[0] if ordering else np.arange(hi - lo)
                F = ppo.Prec(permute(good[s], order), "ic0")
                w = ppo.cg(permute(bad[s], order), b[lo:hi].cpu().numpy()[order], F, tol=1e-300, maxit=3)["x"]
                got = x[lo:hi].cpu().numpy()[order]
                # three steps' rounding: a few eps, magnified by how far alpha and beta lie from one
                assert np.linalg.norm(got - w) <= 1e-11 * np.linalg.norm(w), (step, fail, s)


def test_values_set_under_the_other_order(pp, torch):
    # the permuted copy of an order used before follows values set under another
    systems = [ppo.vardiff2d(s, np.exp(ppo.normal(s * s, 40 + s))) for s in (7, 32)]
    new = scaled(systems, 500)
    b = torch.tensor(np.concatenate([ppo.uniform(len(A[0]) - 1, 5 + s) for s, A in enumerate(systems)]), device="cuda")
    for on_device in (False, True):
        B = pp.BatchedSystems(systems, ordering=1)
        B.set_ordering(0)
        v = np.concatenate([A[2] for A in new])
        B.set_values(torch.tensor(v, device="cuda") if on_device else v)
        B.set_ordering(1)
        F = pp.BatchedSystems(new, ordering=1)
        for (i0, x0), (i1, x1) in zip(solves(torch, B, b), solves(torch, F, b)):
            assert np.array_equal(i0, i1) and torch.equal(x0, x1)


def test_unsorted_rows_are_factored_on_the_host(pp, torch):
    def reversed_rows(A):
        rp, ci, v = A
        back = np.concatenate([np.arange(rp[i], rp[i + 1])[::-1] for i in range(len(rp) - 1)])
        return rp, ci[back], v[back]

    systems = [reversed_rows(ppo.laplacian(9, 8, 1)), ppo.laplacian(7, 6, 1)]
    B = pp.BatchedSystems(systems)
    new = scaled(systems, 300)
    b = torch.ones(B.n, dtype=torch.float64, device="cuda")
    B.set_values(torch.tensor(np.concatenate([A[2] for A in new]), device="cuda"))
    assert B.info().device_refactors == 0
    for (i0, x0), (i1, x1) in zip(solves(torch, B, b), solves(torch, pp.BatchedSystems(new), b)):
        assert np.array_equal(i0, i1) and torch.equal(x0, x1)


def test_refresh_reports_a_failing_pivot(pp, torch):
    from prispack_amd import PrisPackError
    systems = [ppo.laplacian(12, 11, 1), ppo.laplacian(9, 10, 1), ppo.laplacian(8, 8, 1)]
    for ordering in (0, 1):
        B = pp.BatchedSystems(systems, ordering=ordering)
        b = torch.ones(B.n, dtype=torch.float64, device="cuda")
        first = solves(torch, B, b)
        bad = B.v.copy()
        r0 = int(B.row_off[1])
        k = int(B.rp[r0 + 17])
        bad[k:int(B.rp[r0 + 18])] *= np.where(B.ci[k:int(B.rp[r0 + 18])] == r0 + 17, -1.0, 1.0)
        with pytest.raises(PrisPackError) as e:
            B.set_values(torch.tensor(bad, device="cuda"))
        assert "system 1" in str(e.value) and B.info().device_refactors == 0
        B.set_values(torch.tensor(B.v, device="cuda"))  # and good values work again
        assert B.info().device_refactors == 1
        for (i0, x0), (i1, x1) in zip(first, solves(torch, B, b)):
            assert np.array_equal(i0, i1) and torch.equal(x0, x1)
