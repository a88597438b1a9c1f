"""The type-10 and general type-1 kernels (one thread per output value) at the
edges of their launches, through the C ABI against the oracle at 1e-12:
vectors around the powers of two, rectangular bases (more points than
functions), basis levels below the grid level, modes whose matrices are too
large for LDS, one-point terms, column-major and rows layouts."""
import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


@pytest.mark.parametrize("D,L,LB,nq_A,nb_A,nq_B", [(1, 4, 4, 1, 1, 2), (2, 0, 0, 1, 1, 2), (2, 2, 2, 1, 1, 15),
                                                    (3, 4, 4, 3, 2, 2), (3, 5, 3, 2, 2, 1), (5, 3, 3, 1, 1, 2)])
@pytest.mark.parametrize("nvec", [1, 2, 3, 8, 17])
def test_point_kernels_parity(cuda, D, L, LB, nq_A, nb_A, nq_B, nvec):
    import torch
    print(f"case D={D} L={L} LB={LB} nq_A={nq_A} nb_A={nb_A} nq_B={nq_B} nvec={nvec}", flush=True)
    b = E.SG4Basis(D, L, LB, [dict(nq_A=nq_A, nb_A=nb_A, nq_B=nq_B, nb_B=nq_B)] * D)
    o = O.SG4(D, L, LB, nq_A=nq_A, nb_A=nb_A, nq_B=nq_B, nb_B=nq_B)
    rng = np.random.default_rng(10 * D + L + nvec)
    n = o.sum_nq
    V, G = rng.standard_normal(n), rng.standard_normal(n * D * D)
    Jac, sqRJ = 0.5 + rng.random(n), 0.5 + rng.random(n)
    der = [(-1, -1), (0, -1), (D - 1, D - 1)] + ([(0, 1), (1, 0), (-1, 1)] if D > 1 else [])
    F = rng.standard_normal((len(der), n))
    psi = rng.standard_normal((b.nb_ba, nvec))
    for op, ref in ((E.SG4Operator(b, 32, potential=V, type_op=10, G=G, Jac=Jac, sqRJ=sqRJ),
                     o.hpsi(psi, V, None, type_op=10, G=G, Jac=Jac, sqRJ=sqRJ)),
                    (E.SG4Operator(b, 32, potential=("type1", der, F)), o.hpsi_t1g(psi, der, F))):
        assert rel(op.apply_host(psi), ref) < 1e-12                # column-major
        x = torch.tensor(psi, device=cuda)
        y = torch.full_like(x, float("nan"))
        op.apply_rows(x, y)
        torch.cuda.synchronize()
        assert rel(y.cpu().numpy(), ref) < 1e-12
        y.fill_(float("nan"))
        for _ in range(2):
            op.apply_graph(x, y)
        torch.cuda.synchronize()
        assert rel(y.cpu().numpy(), ref) < 1e-12
