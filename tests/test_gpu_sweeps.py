"""The chunked (PP_TRSV_BLOCK) and the strip-wise (PP_TRSV_STRIPS) triangular
sweeps against one launch per level (PP_TRSV_LEVELS, itself pinned to the
oracle): every step shape, all three pairs of diagonal modes, rows of no, one
and many steps, operands whose quotients leave the range of the reciprocal
division.  Equal bit for bit in both precisions: the sweeps do the same
operations in the same order."""
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


def blocks(A, count):
    """count copies of A on the diagonal, every second one cut to half its rows."""
    rp, ci, v = A
    n = len(rp) - 1
    rps, cis, vs, row, nnz = [np.zeros(1, np.int64)], [], [], 0, 0
    for k in range(count):
        m = n // 2 if k % 2 else n
        keep = (np.arange(len(ci)) < rp[m]) & (ci < m)
        cnt = np.add.reduceat(keep[:rp[m]].astype(np.int64), rp[:m].astype(np.int64))
        rps.append(np.cumsum(cnt) + nnz)
        cis.append(ci[keep].astype(np.int64) + row)
        vs.append(v[keep])
        row, nnz = row + m, nnz + int(keep.sum())
    return np.concatenate(rps).astype(np.uint32), np.concatenate(cis).astype(np.uint32), np.concatenate(vs)


def diagonal(d):
    n = len(d)
    return np.arange(n + 1, dtype=np.uint32), np.arange(n, dtype=np.uint32), d


def dense(n):
    a = np.random.default_rng(n).standard_normal((n, n))
    a = a @ a.T + n * np.eye(n)
    return (np.arange(n + 1, dtype=np.uint32) * n, np.tile(np.arange(n, dtype=np.uint32), n), a.ravel())


CASES = {
    # the shapes that the chunked sweep takes: one wavefront with a row on 1 lane of 4 entries (one_row, chain,
    # 2d_short) or 8 (two_levels_long), on 2 of 8 (ilut), on 4 of 4 (narrow, 2d_fill, long_rows, ildlt) or 8
    # (dense); four wavefronts with 4 lanes (3d_wide, blocks) or 1 (two_levels, ilu0) of 4
    # name: matrix, kind, arguments
    "one_row": lambda: (diagonal(np.array([3.0])), "ict", dict(threshold=1e-3)),
    "chain": lambda: (ppo.laplacian(700, 1, 1), "ict", dict(threshold=0.0)),
    "narrow": lambda: (ppo.laplacian(37, 31, 1), "ict", dict(threshold=1e-3)),
    "2d_fill": lambda: (ppo.laplacian(90, 81, 1), "ict", dict(threshold=1e-3)),
    "2d_short": lambda: (ppo.laplacian(101, 90, 1), "ict", dict(threshold=1e-2)),
    "long_rows": lambda: (ppo.laplacian(41, 40, 1), "ict", dict(threshold=0.0)),
    "3d_wide": lambda: (ppo.laplacian(25, 24, 23), "ict", dict(threshold=3e-3)),
    "two_levels": lambda: (ppo.laplacian(113, 90, 1), "ic0", dict(ordering=1)),
    "ildlt": lambda: (ppo.laplacian(61, 54, 1), "ildlt", dict(tolerance=1e-3)),
    "ilut": lambda: (ppo.upwind(19, 18, 17, 20.0, 10.0, 5.0), "ilut", dict(lfill=20, tolerance=1e-2)),
    "ilu0": lambda: (ppo.upwind(19, 18, 17, 20.0, 10.0, 5.0), "ilu0", dict()),
    "blocks": lambda: (blocks(ppo.laplacian(22, 21, 20), 9), "ildlt", dict(tolerance=1e-3)),
    "dense": lambda: (dense(230), "ict", dict(threshold=0.0)),
    "two_levels_long": lambda: (ppo.upwind(27, 27, 27, 20.0, 10.0, 5.0), "ilut",
                                dict(lfill=20, tolerance=1e-2, ordering=1)),
}


def bits(torch, t):
    return t.view(torch.int64 if t.dtype == torch.float64 else torch.int32)


LARGE = {
    # connected parts larger than LDS holds: short rows, two-lane rows, rows of several steps
    "3d_short": lambda: (ppo.laplacian(40, 33, 29), "ict", dict(threshold=1e-2)),
    "3d_long": lambda: (ppo.laplacian(33, 32, 31), "ict", dict(threshold=1e-3)),
    "2d_large": lambda: (ppo.laplacian(211, 190, 1), "ict", dict(threshold=1e-3)),
    "2d_rcm": lambda: (ppo.laplacian(190, 151, 1), "ict", dict(threshold=1e-2, ordering=2)),
    "ildlt_large": lambda: (ppo.laplacian(40, 31, 30), "ildlt", dict(tolerance=3e-3)),
    "ilut_large": lambda: (ppo.upwind(43, 31, 29, 20.0, 10.0, 5.0), "ilut", dict(lfill=20, tolerance=1e-2)),
    "ilu0_large": lambda: (ppo.upwind(43, 31, 29, 20.0, 10.0, 5.0), "ilu0", dict()),
}


@pytest.mark.parametrize("trsv,name", [(3, k) for k in CASES] + [(5, k) for k in [*CASES, *LARGE]])
def test_sweeps_match_levels(pp, torch, trsv, name):
    A, kind, kw = {**CASES, **LARGE}[name]()
    n = len(A[0]) - 1
    print(f"[sweeps] {name} n={n} trsv={trsv}", flush=True)
    M = pp.CSRMatrix(*A)
    cls = {"ict": pp.IncompleteCholesky, "ildlt": pp.IncompleteLDLT, "ilut": pp.IncompleteLU, "ic0": pp.IC0,
           "ilu0": pp.ILU0}[kind]
    P1, P3 = (cls(M, trsv=t, **kw) for t in (1, trsv))
    P1.setup()
    P3.setup()
    if trsv == 5 and n == 1:
        assert P3.info().trsv in (1, 5)
    else:
        assert P1.info().trsv == 1 and P3.info().trsv == trsv
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n)
    x[rng.random(n) < 0.2] = 0.0   # zeros of both signs take the division itself
    x[rng.random(n) < 0.05] = -0.0
    scaled = [x, x * 1e-300, x * 2.0 ** 900, np.where(np.arange(n) == n // 2, np.inf, x)]
    for k, xs in enumerate(scaled):
        for dt in (torch.float64, torch.float32):
            v = torch.tensor(xs, dtype=dt, device="cuda")
            want, got = P1.MInvSolve(v.clone()), torch.full_like(v, 7.0)
            P3.MInvSolve(v, got)
            same = (bits(torch, want) == bits(torch, got)) | (torch.isnan(want) & torch.isnan(got))
            assert bool(same.all()), (name, k, dt, int((~same).sum()))


def test_block_sweep_quotients(pp, torch):
    # a diagonal factor divides twice by each pivot: mantissas and exponents
    # over the whole range, pivots past the reciprocals' range among them
    rng = np.random.default_rng(3)
    n = 20000
    e = rng.integers(-200, 200, n)
    e[::40] = rng.integers(-500, 500, len(e[::40]))
    A = diagonal(rng.uniform(1.0, 2.0, n) * 2.0 ** (2 * e))
    M = pp.CSRMatrix(*A)
    P1, P3 = (pp.IncompleteCholesky(M, 1e-3, trsv=t) for t in (1, 3))
    P1.setup()
    P3.setup()
    assert P3.info().trsv == 3
    for dt, span in ((torch.float64, 1000), (torch.float32, 130)):
        x = rng.uniform(-2.0, 2.0, n) * 2.0 ** rng.integers(-span, span, n)
        v = torch.tensor(x, dtype=dt, device="cuda")
        want, got = P1.MInvSolve(v.clone()), P3.MInvSolve(v.clone())
        same = (bits(torch, want) == bits(torch, got)) | (torch.isnan(want) & torch.isnan(got))
        assert bool(same.all()), int((~same).sum())


@pytest.mark.parametrize("launch", [0, 1])  # captured bodies replayed, bodies launched on the stream
@pytest.mark.parametrize("kind", ["cg", "cg_mixed", "gmres"])
def test_strip_solves_match_levels(pp, torch, kind, launch):
    # whole solves, twice each: the exchange buffers are empty again for every apply
    A = ppo.upwind(33, 31, 29, 20.0, 10.0, 5.0) if kind == "gmres" else ppo.laplacian(33, 31, 29)
    n = len(A[0]) - 1
    M = pp.CSRMatrix(*A)
    b = torch.tensor(ppo.spmv(A, ppo.uniform(n, 4)), device="cuda")
    out = []
    for trsv in (1, 5, 0):
        if kind == "gmres":
            P = pp.IncompleteLU(M, 20, 1e-2, trsv=trsv)
        else:
            P = pp.IncompleteCholesky(M, 1e-2, trsv=trsv, make_f32=kind == "cg_mixed")
        P.setup()
        assert P.info().trsv == trsv or (trsv == 0 and P.info().trsv in (1, 5))
        for _ in range(2):
            if kind == "gmres":
                s = pp.GMRES(n, P, 1e-8, pp.FlexibleGMRES, maxIter=3000)
                s.setRestart(True, 30)
            else:
                s = pp.CG(n, P, pp.FlexibleCG, tol=1e-8, maxIter=1000,
                          precision="mixed" if kind == "cg_mixed" else "fp64")
            s.opts.launch = launch
            x = torch.zeros(n, dtype=torch.float64, device="cuda")
            s.solve(M, b, x)
            assert s.getConvergence()
            out.append((s.getNumIter(), x))
    for it, x in out[1:]:
        assert it == out[0][0] and torch.equal(x, out[0][1])


def _apply_on(ctx, P, x, y):
    import ctypes
    from prispack_amd import _capi
    p = [ctypes.c_void_p(t.data_ptr()) for t in (x, y)]
    ctx.check(_capi.lib().pp_precond_apply(ctx.h, P.h, int(x.dtype.itemsize == 4), *p))


@pytest.mark.parametrize("f32", [False, True])
def test_strips_on_two_contexts_at_once(pp, torch, f32):
    # a preconditioner's applies on two contexts overlap: each context has its
    # own exchange buffers; a second, larger factor makes them grow in between
    import threading
    Ps = []
    for grid in ((40, 33, 29), (48, 40, 33)):
        M = pp.CSRMatrix(*ppo.laplacian(*grid))
        Ps.append([pp.IncompleteCholesky(M, 1e-2, trsv=t, make_f32=f32) for t in (1, 5)])
        for P in Ps[-1]:
            P.setup()
        assert Ps[-1][1].info().trsv == 5
    dt = torch.float32 if f32 else torch.float64
    jobs = []  # (preconditioner, operand, expected, result) by thread
    for k in range(2):
        jobs.append([])
        for i in range(40):
            levels, strips = Ps[int(20 <= i < 30)]
            n = strips.A.n
            x = torch.tensor(ppo.normal(n, 100 * k + i), dtype=dt, device="cuda")
            jobs[k].append((strips, x, levels.MInvSolve(x.clone()), torch.zeros_like(x)))
    torch.cuda.synchronize()
    ctxs = [pp.Context(0), pp.Context(0)]
    gate, failed = threading.Barrier(2), []

    def work(k):
        try:
            gate.wait()
            for P, x, _, y in jobs[k]:
                _apply_on(ctxs[k], P, x, y)
            ctxs[k].sync()
        except Exception as e:
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for k in range(2):
        for i, (_, _, want, got) in enumerate(jobs[k]):
            assert torch.equal(want, got), (k, i)


def test_strips_on_a_context_that_changes_streams(pp, torch):
    # applies queued on one stream after another: they share the context's buffers
    M = pp.CSRMatrix(*ppo.laplacian(40, 33, 29))
    P1, P = (pp.IncompleteCholesky(M, 1e-2, trsv=t) for t in (1, 5))
    P1.setup()
    P.setup()
    ctx = pp.Context(0)
    streams = [torch.cuda.Stream() for _ in range(3)] + [None]
    xs = [torch.tensor(ppo.normal(M.n, 300 + i), device="cuda") for i in range(24)]
    want, ys = [P1.MInvSolve(x.clone()) for x in xs], [torch.zeros_like(x) for x in xs]
    torch.cuda.synchronize()
    for i, (x, y) in enumerate(zip(xs, ys)):
        for k in ([i + 1, i + 2] if i % 5 == 4 else []) + [i]:  # also streams that get no apply in between
            s = streams[k % 4]
            ctx.check(pp._capi.lib().pp_ctx_set_stream(ctx.h, s.cuda_stream if s else None))
        _apply_on(ctx, P, x, y)
    ctx.sync()
    torch.cuda.synchronize()
    ctx.check(pp._capi.lib().pp_ctx_set_stream(ctx.h, None))
    for i, (w, y) in enumerate(zip(want, ys)):
        assert torch.equal(w, y), i


def test_strips_captured(pp, torch):
    # an apply captured on a context that has exchange buffers, and on one
    # that cannot get them inside the capture (level sweeps, the same bits)
    M = pp.CSRMatrix(*ppo.laplacian(40, 33, 29))
    P = pp.IncompleteCholesky(M, 1e-2, trsv=5)
    P.setup()
    x, y = (torch.zeros(M.n, dtype=torch.float64, device="cuda") for _ in range(2))
    stream = torch.cuda.Stream()
    for ready in (True, False):
        ctx = pp.Context(0)
        ctx.check(pp._capi.lib().pp_ctx_set_stream(ctx.h, stream.cuda_stream))
        if ready:
            _apply_on(ctx, P, x, y)
            ctx.sync()
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=stream, capture_error_mode="thread_local"):
            _apply_on(ctx, P, x, y)
        for k in range(4):
            x.copy_(torch.tensor(ppo.normal(M.n, 7 + k), device="cuda"))
            want = P.MInvSolve(x.clone())  # on another context, between the replays
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want), (ready, k)
        del g
