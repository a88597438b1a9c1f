"""Applies that the caller captures into a graph of its own follow a field set
later: the replay acts with the potential that the plan holds then."""
import ctypes as C

import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def noalloc(op, x, y):
    E._capi.check(E.lib().sg4_apply_noalloc(op._h, x.shape[0], C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()),
                                            E.PREC_FP64))


@pytest.mark.parametrize("entry", ["apply", "rows", "noalloc"])
@pytest.mark.parametrize("D,L,nvec", [(4, 5, 1), (4, 5, 3), (6, 6, 4)])
def test_a_captured_apply_follows_the_field(cuda, entry, D, L, nvec):
    import torch
    b, o = E.SG4Basis(D, L), O.SG4(D, L)
    op = E.SG4Operator(b, max_nvec=8)
    assert op.sparse_info()[0]
    side = torch.cuda.Stream()
    E._capi.check(E.lib().sg4_plan_set_stream(op._h, C.c_void_p(side.cuda_stream)))
    psi = np.random.default_rng(nvec).standard_normal((b.nb_ba, nvec))
    x = torch.tensor(psi if entry == "rows" else psi.T.copy(), device=cuda)
    y = torch.full_like(x, float("nan"))
    mu = op.grid_dipole()
    call = {"apply": op.apply, "rows": op.apply_rows, "noalloc": lambda u, v: noalloc(op, u, v)}[entry]
    torch.cuda.synchronize()
    (op.apply if entry == "noalloc" else call)(x, y)      # prepares the plan
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(x, y)
    V, m = o.grid_hh(0.111803), mu.cpu().numpy()
    for field in (None, 0.3, -0.2, None):
        op.set_field(None if field is None else mu, field or 0.0)
        ref = o.hpsi(psi, V + (field or 0.0) * m, -0.5 * np.ones(D))
        for _ in range(2):
            y.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            got = y.cpu().numpy()
            got = got if entry == "rows" else got.T
            assert np.max(np.abs(got - ref)) < 1e-12 * np.max(np.abs(ref)), field
            call(x, y)                                    # eager applies between the replays
            torch.cuda.synchronize()
