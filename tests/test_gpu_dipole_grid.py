"""The field gradient with a dipole operator on a finer grid than H's (the same
packed rows): the dipole operator given is the one that acts."""
import numpy as np
import pytest

import elvibrot_amd as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,L", [(2, 3), (4, 4)])
def test_dipole_operator_on_a_finer_grid(cuda, D, L):
    import torch
    from elvibrot_amd.propagation import ChebyshevPropagator, field_gradient_device
    b, c = E.SG4Basis(D, L, L), E.SG4Basis(D, L + 1, L)
    assert b.nb_ba == c.nb_ba and c.sum_nq > b.sum_nq
    op = E.SG4Operator(b, max_nvec=8)
    mu = op.grid_dipole()
    fine = np.concatenate([c.term_grid(t) for t in range(c.nterms)]).sum(axis=1)
    g = torch.Generator(device=cuda).manual_seed(D)
    r = lambda: torch.randn(1, b.nb_ba, device=cuda, dtype=torch.float64, generator=g)
    psi, target = torch.complex(r(), r()), torch.complex(r(), r())
    psi, target = (x / torch.linalg.norm(x) for x in (psi, target))
    out = []
    for sparse in (True, False):
        op.set_sparse(sparse)
        prop = ChebyshevPropagator(op, 0.05, 0.0, 20.0, mu=mu)
        prop.op_mu = E.SG4Operator(c, max_nvec=8, potential=1.5 * fine, ck=np.zeros(D))
        out.append(field_gradient_device(prop, psi, target, [0.05, -0.1, 0.02], 4, checkpoint_every=2))
    (J, grad), (J0, grad0) = out
    assert abs(J - J0) < 1e-11 * abs(J0)
    assert np.max(np.abs(grad - grad0)) < 1e-11 * np.max(np.abs(grad0))
