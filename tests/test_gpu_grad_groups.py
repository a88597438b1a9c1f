"""Grid-value gradients by the grouped passes against the per-mode ones
(SG4_OPT_GROUPING = 0) on the MI355X: block widths around the item sizes,
phi = psi and phi != psi, terms of one group (1D), of the largest group shapes
(24 points) and of many active modes, absent rows, one-point terms.  Both are
products of two FP64 transforms of at most 16 modes: 1e-13 of the largest
value."""
import numpy as np
import pytest

import elvibrot_amd as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,L,LB,nq_B", [(1, 0, 0, 2), (1, 5, 5, 2), (2, 3, 3, 7), (3, 0, 0, 2), (3, 6, 6, 2), (4, 5, 3, 2),
                                         (6, 6, 6, 2), (12, 3, 3, 1)])
@pytest.mark.parametrize("nvec", [1, 3, 5, 16, 33])
def test_grouped_gradient_equals_per_mode(cuda, D, L, LB, nq_B, nvec):
    import torch
    print(f"case D={D} L={L} LB={LB} nq_B={nq_B} nvec={nvec}", flush=True)
    b = E.SG4Basis(D, L, LB, [dict(nq_B=nq_B)] * D)
    op = E.SG4Operator(b, max_nvec=nvec)
    g = torch.Generator(device=cuda).manual_seed(D + nvec)
    phi, psi = (torch.randn(b.nb_ba, nvec, device=cuda, dtype=torch.float64, generator=g) for _ in range(2))
    out = [torch.full((b.sum_nq, nvec), float("nan"), device=cuda, dtype=torch.float64) for _ in range(4)]
    op.grad_V(phi, psi, out[0])
    op.grad_V(psi, psi, out[1])
    op.set_grouping(False)
    op.grad_V(phi, psi, out[2])
    op.grad_V(psi, psi.clone(), out[3])
    torch.cuda.synchronize()
    for a, r in ((out[0], out[2]), (out[1], out[3])):
        assert (torch.max(torch.abs(a - r)) / torch.max(torch.abs(r))).item() < 1e-13
