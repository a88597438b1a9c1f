"""Chebyshev orders on the sparse matrix where the order kernel changes its
slices (more than 32768 rows) and at its widest blocks, against the term
kernels: the same FP64 recurrences, so equal to the rounding of ~100 applies
(1e-11 relative)."""
import pytest

torch = pytest.importorskip("torch")
import elvibrot_amd as E  # noqa: E402
from elvibrot_amd.propagation import ChebyshevPropagator, field_gradient_device, propagate_device  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes,ns,gradient", [([(8, 6), (4, 4)], 1, True), ([(8, 6), (4, 4)], 2, True),
                                                ([(8, 6), (4, 4)], 4, True), ([(4, 4), (3, 5)], 8, False)])
def test_orders_equal_the_term_kernels(shapes, ns, gradient):
    op = E.SG4Batch([E.SG4Basis(*s) for s in shapes], max_nvec=16)
    assert op.sparse_info()[0] and (op.nb_ba > 32768) == (shapes[0] == (8, 6))
    mu = op.grid_dipole()
    g = torch.Generator(device="cuda").manual_seed(ns)
    r = lambda: torch.randn(ns, op.nb_ba, device="cuda", dtype=torch.float64, generator=g)
    psi, target = torch.complex(r(), r()), torch.complex(r(), r())
    psi, target = (x / torch.linalg.norm(x, dim=1, keepdim=True) for x in (psi, target))
    eps = [0.05, -0.1]
    blocks = list(zip(op.row0[:-1], op.row0[1:]))
    prop = ChebyshevPropagator(op, 0.04, 0.0, 30.0, mu=mu)
    assert prop.nmax * len(eps) >= 24        # applies from which the matrix is built
    out = {}
    for sparse in (True, False):
        op.set_sparse(sparse)
        out[sparse] = [propagate_device(prop, psi, eps, 1)]
        if gradient:
            J, grad = field_gradient_device(prop, psi, target, eps, 1, checkpoint_every=1, blocks=blocks)
            out[sparse] += [torch.tensor([J]), torch.tensor(grad)]
    for a, b in zip(out[True], out[False]):
        assert (torch.max(torch.abs(a - b)) / torch.max(torch.abs(b))).item() < 1e-11
