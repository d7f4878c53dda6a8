"""Bounded waits between workgroups, their limit set to nothing from the host
(pp_ctx_set_wait_limit): every kernel gives up at the first look that finds
nothing and ends normally, the caller gets the documented error or the
fallback's result, and the next call with the usual limit is whole again."""
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
def ctx(torch):
    import prispack_amd as pp
    return pp.Context(0)


def limit(ctx, seconds):
    from prispack_amd import _capi
    ctx.check(_capi.lib().pp_ctx_set_wait_limit(ctx.h, seconds))


def test_limit_arguments(torch, ctx):
    import prispack_amd as pp
    for bad in (-1.0, float("nan"), float("inf")):
        with pytest.raises(pp.PrisPackError) as e:
            limit(ctx, bad)
        assert e.value.status == 1
    limit(ctx, 2.0)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("trsv", [2, 5])  # sync-free, strips
def test_sweep_gives_up(torch, ctx, trsv, f32):
    import prispack_amd as pp
    A = ppo.laplacian(40, 33, 29)
    M = pp.CSRMatrix(*A, ctx=ctx)
    P1, P = (pp.IncompleteCholesky(M, 1e-2, trsv=t, make_f32=f32) for t in (1, trsv))
    P1.setup()
    P.setup()
    assert P.info().trsv == trsv
    x = torch.tensor(ppo.normal(M.n, 3), dtype=torch.float32 if f32 else torch.float64, device="cuda")
    want = P1.MInvSolve(x.clone())
    b = torch.tensor(ppo.normal(M.n, 4), device="cuda")
    for _ in range(2):
        limit(ctx, 0.0)
        with pytest.raises(pp.PrisPackError) as e:
            P.MInvSolve(x.clone())
        assert e.value.status == 2
        S = pp.CG(M.n, P, pp.FlexibleCG, tol=1e-8, maxIter=50, precision="mixed" if f32 else "fp64")
        with pytest.raises(pp.PrisPackError) as e:
            S.solve(M, b, torch.zeros_like(b))
        assert e.value.status == 2
        limit(ctx, 2.0)
        for _ in range(3):
            assert torch.equal(P.MInvSolve(x.clone()), want)
        S.solve(M, b, torch.zeros_like(b))
        assert S.getConvergence()


def test_auto_keeps_the_levels_when_strips_give_up(torch, ctx):
    import prispack_amd as pp
    M = pp.CSRMatrix(*ppo.laplacian(40, 33, 29), ctx=ctx)
    limit(ctx, 0.0)
    P = pp.IncompleteCholesky(M, 1e-2)
    P.setup()
    limit(ctx, 2.0)
    assert P.info().trsv == 1
    x = torch.tensor(ppo.normal(M.n, 3), device="cuda")
    assert bool(torch.isfinite(P.MInvSolve(x)).all())


def test_batch_falls_back(torch, ctx):
    import prispack_amd as pp
    systems = [ppo.vardiff2d(s, np.exp(ppo.normal(s * s, s))) for s in (150, 20, 91)]
    B = pp.BatchedSystems(systems, ctx=ctx, ordering=1)
    xt = np.concatenate([ppo.normal(len(A[0]) - 1, 60 + s) for s, A in enumerate(systems)])
    b = torch.tensor(np.concatenate([ppo.spmv(A, xt[B.row_off[s]:B.row_off[s + 1]]) for s, A in enumerate(systems)]),
                     device="cuda")
    x = [torch.zeros_like(b) for _ in range(4)]
    its = []
    for k, seconds in enumerate((2.0, 0.0, 0.0, 2.0)):
        limit(ctx, seconds)
        its.append(B.solve(b, x[k], precision="mixed", tol=1e-8))
        assert (B.report.batch_tiles > 0) == (seconds > 0)
        assert B.report.converged and B.report.true_relres < 1e-8
    assert torch.equal(x[0], x[3]) and np.array_equal(its[0], its[3])
    assert torch.equal(x[1], x[2]) and np.array_equal(its[1], its[2])
    for s, A in enumerate(systems):
        u, bs = (t[int(B.row_off[s]):int(B.row_off[s + 1])].cpu().numpy() for t in (x[1], b))
        # the solve's test and the rounding of a second FP64 residual
        assert np.linalg.norm(bs - ppo.spmv(A, u)) <= 1.01e-8 * np.linalg.norm(bs), s


def test_strip_apply_returns_before_the_sweep(torch, ctx):
    # the call is asynchronous, as with the level sweeps; a sweep that gives up
    # afterwards is reported by the next call that waits, once
    import ctypes
    import prispack_amd as pp
    from prispack_amd import _capi
    L = _capi.lib()
    M = pp.CSRMatrix(*ppo.laplacian(40, 33, 29), ctx=ctx)
    P = pp.IncompleteCholesky(M, 1e-2, trsv=5)
    P.setup()
    x = torch.tensor(ppo.normal(M.n, 3), device="cuda")
    want, y = P.MInvSolve(x.clone()), torch.zeros_like(x)
    px, py = (ctypes.c_void_p(t.data_ptr()) for t in (x, y))
    stream = torch.cuda.Stream()
    w = torch.ones(8192, 8192, device="cuda")
    torch.cuda.synchronize()
    ctx.check(L.pp_ctx_set_stream(ctx.h, stream.cuda_stream))
    try:
        for seconds in (0.0, 2.0):
            limit(ctx, seconds)
            with torch.cuda.stream(stream):
                for _ in range(20):
                    v = w @ w
            ctx.check(L.pp_precond_apply(ctx.h, P.h, 0, px, py))
            assert not stream.query()
            if seconds == 0.0:
                with pytest.raises(pp.PrisPackError) as e:
                    ctx.sync()
                assert e.value.status == 2 and bool(torch.isnan(y).any())
            ctx.sync()
        assert torch.equal(y, want)
    finally:
        limit(ctx, 2.0)
        torch.cuda.synchronize()
        ctx.check(L.pp_ctx_set_stream(ctx.h, None))


@pytest.mark.parametrize("kind", ["AMSED", "GMSLR"])
def test_multilevel_over_strips(torch, ctx, kind):
    # the subdomain factors wait, not the preconditioner applied: the apply and
    # the set-up fail all the same
    import ctypes
    import prispack_amd as pp
    A = ppo.laplacian(24, 22, 20) if kind == "AMSED" else ppo.upwind(24, 22, 20, 20.0, 10.0, 5.0)
    M = pp.CSRMatrix(*A, ctx=ctx)
    make = lambda trsv: getattr(pp, kind)(M, levels=2, ndom=4, rank=4, trsv=trsv)
    P1, P = make(1), make(5)
    P1.setup()
    P.setup()
    assert P.info().trsv == 5
    x = torch.tensor(ppo.normal(M.n, 3), device="cuda")
    want = P1.MInvSolve(x.clone())
    for _ in range(2):
        limit(ctx, 0.0)
        with pytest.raises(pp.PrisPackError) as e:
            P.MInvSolve(x.clone())
        assert e.value.status == 2
        with pytest.raises(pp.PrisPackError) as e:
            make(5).setup()
        assert e.value.status == 2
        limit(ctx, 2.0)
        for _ in range(2):
            assert torch.equal(P.MInvSolve(x.clone()), want)  # the same set-up, bit for bit
    Q = make(5)  # a set-up behind a failed apply that nobody waited for
    limit(ctx, 0.0)
    y = torch.zeros_like(x)
    torch.cuda.synchronize()
    ctx.check(pp._capi.lib().pp_precond_apply(ctx.h, P.h, 0, *(ctypes.c_void_p(t.data_ptr()) for t in (x, y))))
    limit(ctx, 2.0)
    with pytest.raises(pp.PrisPackError):
        ctx.sync()
    Q.setup()
    assert torch.equal(Q.MInvSolve(x.clone()), want)
