"""FP64 H.psi as one sparse matrix (potentials that are sums of one- and
two-mode functions) through the C ABI on the MI355X: parity with the oracle's
term-by-term sum at the bar of the term kernels (1e-12 of max|H psi|), the
potentials and bases that must keep the term kernels, and the switches
between the two (field, options, graphs)."""
import numpy as np
import pytest

import elvibrot_amd as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-12


def rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


def points(b):
    return np.concatenate([b.term_grid(t) for t in range(b.nterms)])


def pair_potential(q, rng):
    """one-mode Morse-like and two-mode functions of every pair"""
    D = q.shape[1]
    V = 1.5 + np.zeros(len(q))
    for k in range(D):
        V += (1 + 0.1 * k) * (1 - np.exp(-0.3 * q[:, k])) ** 2
    for a in range(D):
        for c in range(a + 1, D):
            if rng.random() < 0.6:
                V += 0.2 * rng.standard_normal() * q[:, a] * q[:, c] + 0.05 * np.cos(q[:, a] - 0.5 * q[:, c])
    return V


@pytest.mark.parametrize("D,L,LB", [(1, 0, 0), (1, 5, 5), (2, 1, 1), (2, 6, 6), (3, 0, 0), (3, 5, 5), (3, 7, 4),
                                    (4, 5, 3), (5, 3, 3), (7, 4, 4)])
@pytest.mark.parametrize("nvec", [1, 2, 4, 7, 16])
def test_pair_potential_parity(cuda, D, L, LB, nvec):
    print(f"case D={D} L={L} LB={LB} nvec={nvec}", flush=True)
    b, o = E.SG4Basis(D, L, LB), O.SG4(D, L, LB)
    rng = np.random.default_rng(100 * D + 10 * L + LB)
    V = pair_potential(points(b), rng)
    ck = -0.5 * (1 + 0.3 * rng.random(D))
    op = E.SG4Operator(b, max_nvec=16, potential=V, ck=ck)
    taken, nnz = op.sparse_info()
    psi = rng.standard_normal((b.nb_ba, nvec))
    ref = o.hpsi(psi, V, ck)
    err = rel(op.apply_host(psi), ref)
    print(f"sparse {taken}, {nnz} entries: {err:.2e}")
    assert err < TOL


@pytest.mark.parametrize("D,L,nvec", [(3, 8, 3), (6, 3, 1), (6, 6, 16), (10, 5, 8), (21, 2, 5), (4, 6, 33)])
def test_henon_heiles_takes_the_sparse_matrix(cuda, D, L, nvec):
    print(f"case D={D} L={L} nvec={nvec}", flush=True)
    b, o = E.SG4Basis(D, L), O.SG4(D, L)
    op = E.SG4Operator(b, max_nvec=64)
    taken, nnz = op.sparse_info()
    assert taken and nnz >= b.nb_ba
    psi = np.random.default_rng(D + L).standard_normal((b.nb_ba, nvec))
    ref = o.hpsi(psi, o.grid_hh(0.111803), -0.5 * np.ones(D))
    assert rel(op.apply_host(psi), ref) < TOL
    op.set_grouping(False)                 # the reference's structure
    assert not op.sparse_info()[0] and rel(op.apply_host(psi), ref) < TOL
    op.set_grouping(True)
    assert op.sparse_info() == (True, nnz)
    op.set_sparse(False)                   # the term kernels of the split path
    assert not op.sparse_info()[0] and rel(op.apply_host(psi), ref) < TOL


def test_modes_of_different_odd_sizes_and_batches(cuda):
    """Modes with their own rules and scales, alone and in a batch of uneven
    instances with one general instance (which keeps the term kernels)."""
    rng = np.random.default_rng(3)
    modes = [dict(nq_B=2), dict(nq_B=4, scaleQ=1.3), dict(nq_B=2, Q0=0.4), dict(nq_B=6)]
    b = E.SG4Basis(4, 3, 3, modes)
    V = pair_potential(points(b), rng)
    ck = -0.5 * (1 + rng.random(4))
    op = E.SG4Operator(b, max_nvec=4, potential=V, ck=ck)
    assert op.split_info()[0] and op.sparse_info()[0]
    psi = rng.standard_normal((b.nb_ba, 3))
    got = op.apply_host(psi)
    op.set_grouping(False)
    assert rel(got, op.apply_host(psi)) < TOL
    bases = [E.SG4Basis(D, L) for D, L in [(4, 4), (2, 5), (6, 3)]]
    Vs = [pair_potential(points(x), rng) for x in bases]
    for general in (False, True):
        if general:
            Vs[2] = Vs[2] + 1e-3 * np.prod(points(bases[2])[:, :3], axis=1)
        op = E.SG4Batch(bases, max_nvec=4, potential=Vs)
        assert op.sparse_info()[0] == (not general)
        psi = rng.standard_normal((op.basis.nb_ba, 2))
        got = op.apply_host(psi)
        for x, v, r0, r1 in zip(bases, Vs, op.row0[:-1], op.row0[1:]):
            assert rel(got[r0:r1], O.SG4(x.D, x.L).hpsi(psi[r0:r1], v, -0.5 * np.ones(x.D))) < TOL


def test_potentials_that_keep_the_term_kernels(cuda):
    """A three-mode coupling of 1e-9, one grid value off, even rules, and NaN."""
    rng = np.random.default_rng(9)
    b, o = E.SG4Basis(5, 4), O.SG4(5, 4)
    q = points(b)
    V0 = pair_potential(q, rng)
    psi = rng.standard_normal((b.nb_ba, 2))
    V1 = V0.copy()
    V1[b.sum_nq // 2] += 1e-9
    for V in (V0 + 1e-9 * q[:, 0] * q[:, 1] * q[:, 2], V1):
        op = E.SG4Operator(b, max_nvec=2, potential=V)
        assert not op.sparse_info()[0]
        assert rel(op.apply_host(psi), o.hpsi(psi, V, -0.5 * np.ones(5))) < TOL
    V1[7] = np.nan
    assert not E.SG4Operator(b, max_nvec=2, potential=V1).sparse_info()[0]
    be = E.SG4Basis(3, 3, 3, [dict(nq_B=1)] * 3)
    op = E.SG4Operator(be, max_nvec=2)
    assert not op.sparse_info()[0]


def test_field_options_and_graphs_switch_paths(cuda):
    """A field adds a term that the matrix does not hold: the term kernels run
    until it is taken back; captured graphs follow."""
    import torch
    D, L = 4, 5
    b, o = E.SG4Basis(D, L), O.SG4(D, L)
    op = E.SG4Operator(b, max_nvec=4)
    V = o.grid_hh(0.111803)
    psi = np.random.default_rng(1).standard_normal((b.nb_ba, 4))
    X = torch.tensor(psi, device=cuda)
    Y = torch.empty_like(X)
    mu = op.grid_dipole()
    for field in (0.0, 0.3, None, 0.2, None):
        if field != 0.0:
            op.set_field(None if field is None else mu, field or 0.0)
        assert op.sparse_info()[0] == (not field)
        ref = o.hpsi(psi, V + (field or 0.0) * mu.cpu().numpy(), -0.5 * np.ones(D))
        for apply in (op.apply_rows, op.apply_graph, op.apply_graph):
            Y.fill_(float("nan"))
            apply(X, Y)
            torch.cuda.synchronize()
            assert rel(Y.cpu().numpy(), ref) < TOL
    op.set_deterministic(True)
    assert not op.sparse_info()[0]
    op.set_deterministic(False)
    E._capi.check(E.lib().sg4_plan_set_henon_heiles(op._h, 0.2))
    ref = o.hpsi(psi, o.grid_hh(0.2), -0.5 * np.ones(D))
    assert op.sparse_info()[0] and rel(op.apply_host(psi), ref) < TOL


@pytest.mark.parametrize("ns", [1, 2, 3, 4])
@pytest.mark.parametrize("dt,steps", [(0.04, 3), (0.06, 3), (0.1, 4)])
def test_propagation_on_the_matrix_equals_the_term_kernels(cuda, ns, dt, steps):
    """Chebyshev steps (odd and even numbers of orders), their field gradient
    and Taylor steps under a field, on the matrix and by the term kernels, on
    a batch: the same maps to FP64 rounding over ~100 applies.  Three states
    have no order kernel and take the term kernels both times."""
    import torch
    from elvibrot_amd.propagation import (ChebyshevPropagator, field_gradient_device, propagate_device,
                                          propagate_taylor_device)
    op = E.SG4Batch([E.SG4Basis(4, 4), E.SG4Basis(3, 5)], max_nvec=16)
    assert op.sparse_info()[0]
    mu = op.grid_dipole()
    g = torch.Generator(device=cuda).manual_seed(ns)
    r = lambda: torch.randn(ns, op.nb_ba, device=cuda, dtype=torch.float64, generator=g)
    psi, target = torch.complex(r(), r()), torch.complex(r(), r())
    psi, target = (x / torch.linalg.norm(x, dim=1, keepdim=True) for x in (psi, target))
    eps = [0.05, -0.1, 0.02]
    blocks = list(zip(op.row0[:-1], op.row0[1:]))
    prop = ChebyshevPropagator(op, dt, 0.0, 20.0, mu=mu)
    out = {}
    for sparse in (True, False):
        op.set_sparse(sparse)
        x = propagate_device(prop, psi, eps, steps)
        J, grad = field_gradient_device(prop, psi, target, eps, steps, checkpoint_every=2, blocks=blocks)
        t, n = propagate_taylor_device(op, psi, dt, 0.0, 20.0, eps, steps, mu=mu)
        t0, n0 = propagate_taylor_device(op, psi, dt, 0.0, 20.0, eps, steps)
        y = torch.empty(op.nb_ba, 2, device=cuda, dtype=torch.float64)
        op.apply_rows(torch.ones_like(y), y)       # no field is left on the plan
        out[sparse] = [x, torch.tensor([J]), torch.tensor(grad), t, torch.tensor(n), t0, torch.tensor(n0), y]
    for a, b in zip(out[True], out[False]):
        if a.is_floating_point() or a.is_complex():
            assert (torch.max(torch.abs(a - b)) / torch.max(torch.abs(b))).item() < 1e-11
        else:
            assert torch.equal(a, b)
    print(f"ns={ns} dt={dt}: {prop.nmax} orders", flush=True)
