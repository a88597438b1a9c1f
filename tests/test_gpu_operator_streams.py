"""An operator set on one stream and applied at once on another (non-blocking)
one, without a synchronisation of the caller's own, against the oracle."""
import ctypes as C

import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def use(op, stream):
    E._capi.check(E.lib().sg4_plan_set_stream(op._h, C.c_void_p(stream.cuda_stream)))


# odd rules: H as one matrix; even ones: the kinetic matrix and the terms
@pytest.mark.parametrize("nq_B", [2, 1])
@pytest.mark.parametrize("nvec", [1, 4])
def test_apply_on_another_stream_than_the_set_up(cuda, nq_B, nvec):
    import torch
    D, L = 6, 5
    modes = [dict(nq_B=nq_B)] * D
    b = E.SG4Basis(D, L, L, modes)
    rng = np.random.default_rng(nq_B)
    q = np.concatenate([b.term_grid(t) for t in range(b.nterms)])
    V = 0.5 * np.sum(q ** 2, axis=1) + 0.1 * q[:, 0] * q[:, 1] ** 2
    ck = -0.5 * np.ones(D)
    psi = rng.standard_normal((b.nb_ba, nvec))
    x = torch.tensor(psi.T.copy(), device=cuda)
    ref = O.SG4(D, L, L, nq_B=nq_B).hpsi(psi, V, ck)
    side = torch.cuda.Stream()
    for _ in range(5):
        y = torch.full_like(x, float("nan"))
        torch.cuda.synchronize()
        op = E.SG4Operator(b, max_nvec=4, potential=V, ck=ck)   # on the default stream
        use(op, side)
        op.apply(x, y)
        torch.cuda.synchronize()
        assert op.sparse_info()[0] == (nq_B == 2)
        assert np.max(np.abs(y.cpu().numpy().T - ref)) < 1e-12 * np.max(np.abs(ref))


def test_field_gradient_with_the_dipole_on_another_stream(cuda):
    import torch
    from elvibrot_amd.propagation import ChebyshevPropagator, field_gradient_device
    b = E.SG4Basis(4, 4)
    op = E.SG4Operator(b, max_nvec=8)
    mu = op.grid_dipole()
    g = torch.Generator(device=cuda).manual_seed(1)
    r = lambda: torch.randn(1, b.nb_ba, device=cuda, dtype=torch.float64, generator=g)
    psi, target = torch.complex(r(), r()), torch.complex(r(), r())
    psi, target = (x / torch.linalg.norm(x) for x in (psi, target))
    got = []
    for side in (None, torch.cuda.Stream()):
        op.set_sparse(False)                 # the dipole operator is applied for itself
        prop = ChebyshevPropagator(op, 0.05, 0.0, 20.0, mu=mu)
        torch.cuda.synchronize()
        mu_op = E.SG4Operator(b, max_nvec=8, potential=mu.cpu().numpy(), ck=np.zeros(4),
                              stream=None if side is None else side.cuda_stream)
        prop.op_mu = mu_op
        got.append(field_gradient_device(prop, psi, target, [0.05, -0.1], 2))
    assert abs(got[0][0] - got[1][0]) < 1e-12
    assert np.max(np.abs(np.array(got[0][1]) - np.array(got[1][1]))) < 1e-12
