"""Values set from a device tensor stay on the device until something reads
them on the host: every such reader sees the new ones, the same bits as after
the same values set from the host."""
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


def _view(pp, torch, A, x):
    return np.asarray(A.host()[2]), np.asarray(A.v)


def _transpose(pp, torch, A, x):
    y = torch.zeros_like(x)
    A.transMatPVec(x, y)
    return (y.cpu().numpy(),)


def _apply(M, A, x, torch):
    M.setup()
    y = torch.zeros_like(x)
    M.MInvSolve(x, y)
    return (y.cpu().numpy(),)


def _threshold(pp, torch, A, x):  # factored on the host
    return _apply(pp.IncompleteCholesky(A, 1e-2), A, x, torch)


def _level0(pp, torch, A, x):  # factored on the device, then read on the host
    M = pp.IC0(A, ordering=1)
    return _apply(M, A, x, torch) + M.factor(0)


def _multilevel(pp, torch, A, x):
    return _apply(pp.AMSED(A, levels=2, ndom=4, rank=8), A, x, torch)


@pytest.mark.parametrize("read", [_view, _transpose, _threshold, _level0, _multilevel])
def test_host_reader_after_device_values(pp, torch, read):
    P = ppo.laplacian(13, 12, 11)
    n = len(P[0]) - 1
    x = torch.tensor(ppo.uniform(n, 5), device="cuda")
    d = 1.0 + 0.25 * ppo.uniform(n, 6)  # D P D: as definite as P
    rows = np.repeat(np.arange(n), np.diff(np.asarray(P[0], np.int64)))
    v2 = np.asarray(P[2]) * d[rows] * d[np.asarray(P[1], np.int64)]
    got = []
    for on_device in (False, True):
        A = pp.CSRMatrix(*P)
        _transpose(pp, torch, A, x)  # the old values were read before
        vals = torch.tensor(v2, device="cuda") if on_device else v2.copy()
        A.set_values(vals)
        vals[:] = 0  # the caller's array is its own again
        got.append(read(pp, torch, A, x))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    if read is _view:
        assert np.array_equal(got[1][0], v2)
