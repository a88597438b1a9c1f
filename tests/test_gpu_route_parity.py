"""Parity with the oracle on a stated route: the sparse matrix for pair potentials
(also with a basis level below the grid level), and the FP64 term kernels with
atomics and with row sums at 10D L=8 x16, whose operator takes the matrix
otherwise."""
import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,L,LB", [(1, 5, 5), (2, 6, 6), (3, 0, 0), (3, 5, 5), (3, 7, 4), (4, 5, 3), (5, 3, 3), (7, 4, 4)])
@pytest.mark.parametrize("nvec", [1, 5, 16])
def test_pair_potentials_take_the_matrix(cuda, D, L, LB, nvec):
    print(f"case D={D} L={L} LB={LB} nvec={nvec}", flush=True)
    b, o = E.SG4Basis(D, L, LB), O.SG4(D, L, LB)
    rng = np.random.default_rng(D * 100 + L * 10 + LB)
    q = np.concatenate([b.term_grid(t) for t in range(b.nterms)])
    V = 0.7 + sum((1 + 0.2 * k) * (1 - np.exp(-0.3 * q[:, k])) ** 2 for k in range(D))
    for a in range(D):
        for c in range(a + 1, D):
            V = V + 0.1 * (a - c) * q[:, a] * q[:, c] ** 2 + 0.05 * np.cos(q[:, a] - 0.4 * q[:, c])
    ck = -0.5 * (1 + 0.3 * rng.random(D))
    op = E.SG4Operator(b, max_nvec=16, potential=V, ck=ck)
    taken, nnz = op.sparse_info()
    assert taken and nnz >= b.nb_ba
    psi = rng.standard_normal((b.nb_ba, nvec))
    ref = o.hpsi(psi, V, ck)
    assert np.max(np.abs(op.apply_host(psi) - ref)) < 1e-12 * np.max(np.abs(ref))


def test_fp64_term_kernels_at_10d_against_the_extended_oracle(cuda):
    """The bars of the deterministic parity test of this workload: 2-norm 1e-12 a
    vector, and 4 eps of max_e sum_t |W_t r_t|; the order of an FP64 sum over the
    terms adds at most their number of roundings, sqrt of it as independent ones."""
    import torch
    D, L, nvec = 10, 8, 16
    b, o = E.SG4Basis(D, L), O.SG4(D, L)
    op = E.SG4Operator(b, max_nvec=nvec)
    op.set_sparse(False)
    psi = np.random.default_rng(2026).standard_normal((b.nb_ba, nvec))
    V = o.grid_hh(0.111803)
    ref = o.hpsi_ld(psi, V, -0.5 * np.ones(D))
    bound = np.max(o.absbound(psi, V, np.zeros(D)))
    eps = np.finfo(np.float64).eps
    x = torch.tensor(psi, device=cuda)
    y = torch.empty_like(x)
    for entry, name in ((op.apply_rows, "atomics"), (op.apply_graph, "row sums"), (op.apply_rows, "row sums")):
        y.fill_(float("nan"))
        entry(x, y)
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        e2 = np.max(np.linalg.norm(got - ref, axis=0) / np.linalg.norm(ref, axis=0))
        r = np.max(np.abs(got - ref)) / (eps * bound)
        print(f"10D L=8 x16 {name}: worst 2-norm {e2:.2e}, max|err| / (eps max bound) {r:.2f}", flush=True)
        assert e2 < 1e-12 and r < 4
