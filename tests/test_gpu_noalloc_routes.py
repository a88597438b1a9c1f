"""One sg4_apply prepares the allocation-free entry for its width and precision,
whichever route (sparse matrix or term kernels) the calls before and after a
field take."""
import ctypes as C

import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nvec", [1, 3, 8])
@pytest.mark.parametrize("D,L", [(4, 5), (6, 6)])
def test_noalloc_after_the_route_changed(cuda, D, L, nvec):
    import torch
    b, o = E.SG4Basis(D, L), O.SG4(D, L)
    psi = np.random.default_rng(nvec).standard_normal((b.nb_ba, nvec))
    x = torch.tensor(psi.T.copy(), device=cuda)
    y = torch.empty_like(x)

    def noalloc(op, field, m):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        E._capi.check(E.lib().sg4_apply_noalloc(op._h, nvec, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()),
                                                E.PREC_FP64))
        torch.cuda.synchronize()
        ref = o.hpsi(psi, o.grid_hh(0.111803) + field * m, -0.5 * np.ones(D))
        assert np.max(np.abs(y.cpu().numpy().T - ref)) < 1e-12 * np.max(np.abs(ref))

    for first in (0.0, 0.4):             # the preparing apply: without and under a field
        op = E.SG4Operator(b, max_nvec=8)
        mu = op.grid_dipole()
        m = mu.cpu().numpy()
        if first:
            op.set_field(mu, first)
        op.apply(x, y)
        noalloc(op, first, m)
        op.set_field(mu, 0.3)
        noalloc(op, 0.3, m)
        op.set_field(None, 0.0)
        assert op.sparse_info()[0]
        noalloc(op, 0.0, m)
        # a launch set for another width and precision changes nothing here
        op.set_config(2, E.PREC_F32, nthreads=512)
        noalloc(op, 0.0, m)
        op.set_sparse(False)
        noalloc(op, 0.0, m)
