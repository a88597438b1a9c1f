"""A propagation leaves the plan without a field, also when it ends with an
error and whichever route (matrix or term kernels) it took."""
import ctypes as C

import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparse", [True, False])
@pytest.mark.parametrize("with_mu", [True, False])
@pytest.mark.parametrize("npoly,max_norm2", [(2, 0.0), (60, 1e-3)])
def test_field_is_taken_back_on_errors(cuda, sparse, with_mu, npoly, max_norm2):
    import torch
    b, o = E.SG4Basis(4, 5), O.SG4(4, 5)
    op = E.SG4Operator(b, max_nvec=4)
    op.set_sparse(sparse)
    mu = op.grid_dipole()
    x = torch.randn(b.nb_ba, 2, device=cuda, dtype=torch.float64)
    x /= torch.linalg.norm(x)
    eps = np.full(8, 0.1)
    prm = E._capi.TaylorParams()
    prm.dt, prm.E0, prm.npoly, prm.poly_tol, prm.max_norm2 = 0.02, 0.0, npoly, 1e-20, max_norm2
    prm.nseg, prm.steps_per_seg, prm.eps, prm.prec = 8, 1, eps.ctypes.data_as(E._capi.D_P), E.PREC_FP64
    op.set_field(mu, 0.3)
    rc = E.lib().sg4_taylor_propagate(op._h, C.c_void_p(mu.data_ptr() if with_mu else None), 1,
                                      C.c_void_p(x.data_ptr()), C.byref(prm), None)
    assert rc == E._capi.ERR_STATE
    psi = np.random.default_rng(0).standard_normal((b.nb_ba, 2))
    ref = o.hpsi(psi, o.grid_hh(0.111803), -0.5 * np.ones(4))
    assert np.max(np.abs(op.apply_host(psi) - ref)) < 1e-12 * np.max(np.abs(ref))
