"""sg4_block_combine on both sides of the lines between its two kernels (matrix
cores, one thread per column): few rows of X over long rows, few rows of Y beyond
the caches."""
import ctypes as C

import numpy as np
import pytest

import elvibrot_amd as E

pytestmark = pytest.mark.gpu


def ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("n,k,d", [(n, k, d) for n in ((1 << 19) - 1, 1 << 19) for k, d in
                                   ((1, 1), (4, 8), (5, 9), (16, 8), (17, 8), (40, 7), (64, 9))] +
                         [(800001, 4, 59), (800001, 4, 61), (800001, 5, 61), (1000, 2, 47), (1000, 2, 48), (999, 1, 124),
                          (1000, 3, 48)])
@pytest.mark.parametrize("beta", [0.0, 1.0, -0.5])
def test_both_kernels(cuda, n, k, d, beta):
    import torch
    op = E.SG4Operator(E.SG4Basis(3, 2), max_nvec=1)
    g = torch.Generator(device=cuda).manual_seed(k * 1000 + d)
    X = torch.randn(d, n, device=cuda, dtype=torch.float64, generator=g)
    U = torch.randn(k, d, device=cuda, dtype=torch.float64, generator=g)
    Y = torch.randn(k, n, device=cuda, dtype=torch.float64, generator=g)
    ref, mag = U @ X + beta * Y, U.abs() @ X.abs() + Y.abs()
    if beta == 0.0:
        Y.fill_(float("nan"))                    # is not read
    E._capi.check(E.lib().sg4_block_combine(op._h, k, d, n, ptr(U), ptr(X), n, beta, ptr(Y), n))
    # two FP64 sums of d + 1 terms
    assert bool(torch.all((Y - ref).abs() <= 2 * (d + 8) * 2.3e-16 * mag))
