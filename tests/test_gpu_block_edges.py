"""The matrix-core block products at the edges of their tiles against numpy:
inner dimensions around the 16- and 32-column steps, row counts around the
16-row tiles and the tile groups, wide against narrow blocks both ways, the
smallest and the largest U in LDS, and NaN confined to its own outputs."""
import ctypes as C

import numpy as np
import pytest

import elvibrot_amd as E

pytestmark = pytest.mark.gpu


def ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 64, 1000])
@pytest.mark.parametrize("m,q", [(1, 1), (15, 17), (16, 16), (17, 1), (1, 40), (33, 65), (64, 31), (5, 124)])
def test_gram_edges(cuda, n, m, q):
    import torch
    op = E.SG4Operator(E.SG4Basis(3, 2), max_nvec=1)
    g = torch.Generator(device=cuda).manual_seed(n * 1000 + m + q)
    A = torch.randn(m, n + 3, device=cuda, dtype=torch.float64, generator=g)[:, 1:1 + n]
    B = torch.randn(q, n + 1, device=cuda, dtype=torch.float64, generator=g)[:, :n]
    work = torch.empty(2048 * m * q, device=cuda, dtype=torch.float64)
    out = torch.full((m, q), float("nan"), device=cuda, dtype=torch.float64)
    call = lambda: E._capi.check(E.lib().sg4_block_gram(op._h, m, q, n, ptr(A), A.stride(0), ptr(B), B.stride(0),
                                                        ptr(out), ptr(work), work.numel()))
    call()
    ref = A.cpu().numpy() @ B.cpu().numpy().T
    scale = np.abs(A.cpu().numpy()) @ np.abs(B.cpu().numpy()).T
    assert np.all(np.abs(out.cpu().numpy() - ref) <= (n + 8) * 2.3e-16 * scale)
    A[m - 1, n - 1] = float("nan")
    call()
    got = out.cpu().numpy()
    assert np.isnan(got[m - 1]).all() and not np.isnan(got[:m - 1]).any()


@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 1000])
@pytest.mark.parametrize("k,d", [(1, 1), (16, 4), (17, 5), (32, 16), (33, 19), (65, 63), (128, 64), (1, 8192), (1, 500)])
def test_combine_edges(cuda, n, k, d):
    import torch
    op = E.SG4Operator(E.SG4Basis(3, 2), max_nvec=1)
    g = torch.Generator(device=cuda).manual_seed(n * 100 + k + d)
    X = torch.randn(d, n + 5, device=cuda, dtype=torch.float64, generator=g)[:, 2:2 + n]
    U = torch.randn(k, d, device=cuda, dtype=torch.float64, generator=g)
    Yb = torch.full((k, n + 2), 7.0, device=cuda, dtype=torch.float64)
    Y = Yb[:, 1:1 + n]
    Y.fill_(0.5)
    E._capi.check(E.lib().sg4_block_combine(op._h, k, d, n, ptr(U), ptr(X), X.stride(0), -2.0, ptr(Y), Y.stride(0)))
    u, x = U.cpu().numpy(), X.cpu().numpy()
    assert np.all(np.abs(Y.cpu().numpy() - (u @ x - 1.0)) <= (d + 8) * 2.3e-16 * (np.abs(u) @ np.abs(x) + 1.0))
    assert torch.all(Yb[:, 0] == 7.0) and torch.all(Yb[:, n + 1] == 7.0)
