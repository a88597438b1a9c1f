"""A propagation builds the matrix with the dipole's values only where its orders
save what that takes: short ones of many coupled modes are not slower than on the
term kernels."""
import pytest

torch = pytest.importorskip("torch")
import elvibrot_amd as E  # noqa: E402
from elvibrot_amd.propagation import ChebyshevPropagator, propagate_device  # noqa: E402
from test_gpu_long_rows import median_us, pairs  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,L,steps", [(32, 2, 1), (32, 2, 4), (21, 2, 2), (6, 3, 1)])
def test_short_propagations(D, L, steps):
    op = pairs(D, L, 4)
    prop = ChebyshevPropagator(op, 0.02, 0.0, 40.0, mu=op.grid_dipole())
    psi = torch.randn(1, op.nb_ba, device="cuda", dtype=torch.complex128)
    psi /= torch.linalg.norm(psi)
    us = {}
    for sparse in (True, False):
        op.set_sparse(sparse)
        us[sparse] = median_us(lambda: propagate_device(prop, psi, [0.01, 0.02, 0.0], steps), 3)
    n = 3 * steps * (prop.nmax - 1)
    print(f"{D}D L={L}, {n} orders: with the matrix {us[True]:.0f} us, term kernels {us[False]:.0f} us", flush=True)
    assert us[True] < 1.25 * us[False]


def test_long_propagations_take_the_matrix():
    op = pairs(6, 4, 4)
    prop = ChebyshevPropagator(op, 0.02, 0.0, 40.0, mu=op.grid_dipole())
    psi = torch.randn(1, op.nb_ba, device="cuda", dtype=torch.complex128)
    us = {}
    for sparse in (True, False):
        op.set_sparse(sparse)
        us[sparse] = median_us(lambda: propagate_device(prop, psi, [0.01, 0.02, 0.0], 10), 3)
    print(f"with the matrix {us[True]:.0f} us, term kernels {us[False]:.0f} us", flush=True)
    assert us[True] < 0.8 * us[False]
