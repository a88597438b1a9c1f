"""Many modes all coupled in pairs at a low level: a few packed rows couple to
almost all others.  The products and Chebyshev orders of such matrices against the
one-vector product and the term kernels, and their times against the term kernels."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import elvibrot_amd as E  # noqa: E402
from elvibrot_amd.propagation import ChebyshevPropagator, field_gradient_device, propagate_device  # noqa: E402

pytestmark = pytest.mark.gpu


def pairs(D, L, max_nvec):
    b = E.SG4Basis(D, L)
    q = np.concatenate([b.term_grid(t) for t in range(b.nterms)])
    V = 0.5 * np.sum(q ** 2, axis=1)
    for a in range(D):
        for c in range(a + 1, D):
            V = V + 0.05 * np.cos(q[:, a] - 0.4 * q[:, c])
    op = E.SG4Operator(b, max_nvec=max_nvec, potential=V, ck=-0.5 * np.ones(D))
    assert op.sparse_info()[0]
    return op


# a row of n <= 2200 entries in another order: n 2^-52 sum|h x| at most, sum|h x|
# below ~n max|h| max|x| / 10 and max|y| above max|h| max|x|: 2200 2^-52 220 = 1e-10;
# the roundings are independent, a tenth of their number's bound and less: 1e-11
@pytest.mark.parametrize("D,L", [(7, 4), (12, 3), (32, 2)])
def test_widths_equal_single_vectors(D, L):
    op = pairs(D, L, 48)
    g = torch.Generator(device="cuda").manual_seed(D)
    x = torch.randn(op.nb_ba, 48, device="cuda", dtype=torch.float64, generator=g)
    one = torch.empty_like(x)
    for v in range(48):
        c = x[:, v:v + 1].contiguous()
        one[:, v:v + 1] = op.apply_rows(c, torch.empty_like(c))
    tol = 1e-11 * float(one.abs().max())
    for w in (2, 3, 4, 5, 7, 8, 9, 13, 16, 24, 32, 33, 40, 48):
        c = x[:, :w].contiguous()
        y = op.apply_rows(c, torch.full_like(c, float("nan")))
        assert float((y - one[:, :w]).abs().max()) <= tol, ("rows", w)
        t = c.t().contiguous()
        z = op.apply(t, torch.full_like(t, float("nan")))
        assert float((z.t() - one[:, :w]).abs().max()) <= tol, ("columns", w)


@pytest.mark.parametrize("D,L", [(7, 4), (12, 3)])
@pytest.mark.parametrize("ns", [1, 2, 4, 8])
def test_orders_equal_the_term_kernels(D, L, ns):
    op = pairs(D, L, 16)
    mu = op.grid_dipole()
    g = torch.Generator(device="cuda").manual_seed(ns)
    r = lambda: torch.randn(ns, op.nb_ba, device="cuda", dtype=torch.float64, generator=g)
    psi, target = torch.complex(r(), r()), torch.complex(r(), r())
    psi, target = (x / torch.linalg.norm(x, dim=1, keepdim=True) for x in (psi, target))
    eps = [0.05, -0.1, 0.03]
    prop = ChebyshevPropagator(op, 0.04, 0.0, 60.0, mu=mu)
    out = {}
    for sparse in (True, False):
        op.set_sparse(sparse)
        out[sparse] = [propagate_device(prop, psi, eps, 4)]
        if ns <= 4:
            J, grad = field_gradient_device(prop, psi, target, eps, 4, checkpoint_every=2)
            out[sparse] += [torch.tensor([J]), torch.tensor(grad)]
    for a, b in zip(out[True], out[False]):
        assert (torch.max(torch.abs(a - b)) / torch.max(torch.abs(b))).item() < 1e-11


def median_us(f, n, repeats=7):
    for _ in range(n):
        f()
    times = []
    for _ in range(repeats):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(n):
            f()
        e1.record()
        torch.cuda.synchronize()
        times.append(e0.elapsed_time(e1) * 1e3 / n)
    return sorted(times)[repeats // 2]


# measured here 0.4 to 0.7 of the term kernels; half as long again would be a fault
@pytest.mark.parametrize("D,L,nvec", [(32, 2, 8), (32, 2, 16), (21, 2, 24), (16, 3, 8), (12, 3, 16)])
def test_the_matrix_is_not_slower_than_the_term_kernels(D, L, nvec):
    op = pairs(D, L, 32)
    x = torch.randn(nvec, op.nb_ba, device="cuda", dtype=torch.float64)
    y = torch.empty_like(x)
    us = {}
    for sparse in (True, False):
        op.set_sparse(sparse)
        us[sparse] = median_us(lambda: op.apply(x, y), 50)
    print(f"{D}D L={L} x{nvec}: matrix {us[True]:.1f} us, term kernels {us[False]:.1f} us", flush=True)
    assert us[True] < 1.2 * us[False]
