"""A field set inside a graph of the caller: the plan's potential changes when the
graph is replayed, and every later apply acts with the potential as it is then."""
import ctypes as C

import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_applies_after_the_replay_of_a_captured_field(cuda):
    import torch
    D, L, nvec = 4, 5, 4
    b, o = E.SG4Basis(D, L), O.SG4(D, L)
    op = E.SG4Operator(b, max_nvec=4)
    assert op.sparse_info()[0]
    side = torch.cuda.Stream()
    E._capi.check(E.lib().sg4_plan_set_stream(op._h, C.c_void_p(side.cuda_stream)))
    psi = np.random.default_rng(5).standard_normal((b.nb_ba, nvec))
    x = torch.tensor(psi, device=cuda)
    y = torch.empty_like(x)
    mu = op.grid_dipole()
    V, m = o.grid_hh(0.111803), mu.cpu().numpy()
    torch.cuda.synchronize()
    op.set_field(mu, 0.1)                  # the plan keeps the field-free potential from here on
    op.set_field(None, 0.0)
    for entry in (op.apply_rows, op.apply_graph):
        entry(x, y)

    def check(field, what):
        ref = o.hpsi(psi, V + field * m, -0.5 * np.ones(D))
        for entry in (op.apply_rows, op.apply_graph, op.apply_graph):
            y.fill_(float("nan"))
            torch.cuda.synchronize()
            entry(x, y)
            torch.cuda.synchronize()
            assert np.max(np.abs(y.cpu().numpy() - ref)) < 1e-12 * np.max(np.abs(ref)), what

    check(0.0, "no field")
    torch.cuda.synchronize()
    graphs = {}
    for f in (0.3, 0.0):
        graphs[f] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graphs[f], stream=side):
            op.set_field(mu if f else None, f)
    op.set_field(None, 0.0)
    check(0.0, "captured, not replayed")
    for _ in range(2):
        for f in (0.3, 0.0):
            graphs[f].replay()
            check(f, f"replayed {f}")
    op.set_field(mu, -0.2)
    check(-0.2, "set by a plain call")
    E._capi.check(E.lib().sg4_plan_set_henon_heiles(op._h, 0.111803))
    assert op.sparse_info()[0]
    check(0.0, "a new operator")
