"""Products with the sparse matrix at every block width that has a kernel of its
own (pairs of columns, column blocks of wider ones, in place and staged
column-major blocks) against the one-vector kernel.  Both are FP64 sums of the
same row entries in another order: a row of n <= 100 entries differs by at most
n 2^-52 sum|h x|, and sum|h x| stays below ~10 max|y| here: 1e-12 max|y| with a
cushion."""
import pytest

torch = pytest.importorskip("torch")
import elvibrot_amd as E  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,L", [(2, 2), (4, 4), (6, 6), (8, 6)])
def test_widths_equal_single_vectors(D, L):
    op = E.SG4Operator(E.SG4Basis(D, L), max_nvec=48)
    assert op.sparse_info()[0]
    g = torch.Generator(device="cuda").manual_seed(D)
    x = torch.randn(op.nb_ba, 48, device="cuda", dtype=torch.float64, generator=g)
    one = torch.empty_like(x)
    for v in range(48):
        c = x[:, v:v + 1].contiguous()
        one[:, v:v + 1] = op.apply_rows(c, torch.empty_like(c))
    tol = 1e-12 * float(one.abs().max())
    for w in (2, 3, 4, 5, 6, 8, 12, 16, 24, 32, 40, 48):
        c = x[:, :w].contiguous()
        y = op.apply_rows(c, torch.full_like(c, float("nan")))
        assert float((y - one[:, :w]).abs().max()) <= tol, ("rows", w)
        t = c.t().contiguous()
        z = op.apply(t, torch.full_like(t, float("nan")))
        assert float((z.t() - one[:, :w]).abs().max()) <= tol, ("columns", w)
