"""The kernels that store the terms' results and the row sums, on a plan whose
map is inverted (its graph entry does that at once), with potentials that couple
all modes, against the oracle."""
import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# the bars of the precision modes against the oracle, of max|H psi|: FP64 as for
# the atomics (1e-12); the reduced modes round V, the matrices and the vectors to
# 24 bits and pass ~2 D contractions of up to n terms on each, and the Smolyak sum
# has partial sums of up to ~1e3 times the result: 2 D n 2^-24 1e3 = 1e-2 is the
# worst case; the roundings are independent, sqrt(2 D n nterms) instead of their
# number, which stays below 1e-4 here
TOL = {E.PREC_FP64: 1e-12, E.PREC_F32: 1e-4, E.PREC_F32X2: 1e-4}


@pytest.mark.parametrize("prec", [E.PREC_FP64, E.PREC_F32, E.PREC_F32X2])
@pytest.mark.parametrize("D,L,LB,widths", [(6, 6, 6, (1, 2, 5, 16, 24)), (5, 8, 7, (3, 8)), (7, 6, 5, (1, 4))])
def test_sums_against_the_oracle(cuda, D, L, LB, widths, prec):
    import torch
    b, o = E.SG4Basis(D, L, LB), O.SG4(D, L, LB)
    assert b.sum_nb >= 1 << 16
    rng = np.random.default_rng(D * 10 + L)
    q = np.concatenate([b.term_grid(t) for t in range(b.nterms)])
    V = 0.5 * np.sum(q ** 2, axis=1) + 0.05 * np.sin(q[:, 0] + q[:, 1] * q[:, 2]) + 0.1 * np.cos(q.sum(axis=1))
    ck = -0.5 * (1 + 0.2 * rng.random(D))
    op = E.SG4Operator(b, max_nvec=max(widths), potential=V, ck=ck)
    assert op.split_info()[0] and not op.sparse_info()[0]
    x0 = torch.zeros(b.nb_ba, max(widths), device=cuda, dtype=torch.float64)
    op.apply_graph(x0, torch.empty_like(x0), prec)
    for w in widths:
        psi = rng.standard_normal((b.nb_ba, w))
        x = torch.tensor(psi, device=cuda)
        y = torch.full_like(x, float("nan"))
        ref = o.hpsi(psi, V, ck)
        for entry in (op.apply_rows, op.apply_graph):
            y.fill_(float("nan"))
            entry(x, y, prec)
            torch.cuda.synchronize()
            err = np.max(np.abs(y.cpu().numpy() - ref)) / np.max(np.abs(ref))
            print(f"{D} {L} {LB} x{w} prec {prec}: {err:.2e}", flush=True)
            assert err < TOL[prec]
