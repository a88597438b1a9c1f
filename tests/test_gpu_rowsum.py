"""Sum of the terms' results row by row (the plain applies of term sets of
2^16 places and more) against the exact fixed-point accumulation of the same
kernels' results: per-term values are the same numbers in both, so the two
differ by the rounding of one FP64 sum per row.  A row is in at most n terms
and its partial sums exceed the largest result by at most ~1e3, so that is
below n 2^-53 1e3 max|y|."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
import elvibrot_amd as E  # noqa: E402

pytestmark = pytest.mark.gpu


def tol(n, ref):
    return n * 2.0 ** -53 * 1e3 * float(ref.abs().max())


def pair(op, x, prec):
    y, z = torch.empty_like(x), torch.empty_like(x)
    op.set_deterministic(False)
    for _ in range(9):            # the first applies of a plan use atomics
        op.apply_rows(x, y, prec)
    op.set_deterministic(True)
    op.apply_rows(x, z, prec)
    op.set_deterministic(False)
    torch.cuda.synchronize()
    return y, z


# 6D L=6: one-workgroup-wide items of 64, 128 and 256 threads, odd widths, rows
# in one and in many segments; 8D L=8: terms beyond the LDS budget, classes kept
# on one XCD; 4D L=11 (wide 1-D bases, one- and two-mode groups)
@pytest.mark.parametrize("prec", [E.PREC_FP64, E.PREC_F32, E.PREC_F32X2])
@pytest.mark.parametrize("D,L,widths", [(6, 6, (1, 2, 3, 5, 8, 16, 17, 24, 33)), (8, 8, (1, 8)), (4, 11, (1, 6, 16))])
def test_row_sums_match_exact_accumulation(D, L, widths, prec):
    b = E.SG4Basis(D, L)
    assert b.sum_nb >= 1 << 16
    op = E.SG4Operator(b, max_nvec=max(widths))
    op.set_sparse(False)
    g = torch.Generator(device="cuda").manual_seed(D * 100 + L)
    for w in widths:
        x = torch.randn(op.nb_ba, w, device="cuda", dtype=torch.float64, generator=g)
        y, z = pair(op, x, prec)
        assert float((y - z).abs().max()) <= tol(b.nterms, z), (w, prec)


@pytest.mark.parametrize("prec", [E.PREC_FP64, E.PREC_F32, E.PREC_F32X2])
def test_block_of_a_batch_graphs_and_streams(prec):
    """The block of results belongs to a stream and grows with the width: an
    instance batch, the plan's own graphs replayed with wider applies between,
    a change of the stream, a capture by the caller (it keeps the atomics) and
    the allocation-free entry all give the plain result."""
    bs = [E.SG4Basis(6, 6), E.SG4Basis(5, 6), E.SG4Basis(6, 5)]
    op = E.SG4Batch(bs, max_nvec=16)
    op.set_sparse(False)
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(op.nb_ba, 4, device="cuda", dtype=torch.float64, generator=gen)
    wide = torch.randn(op.nb_ba, 16, device="cuda", dtype=torch.float64, generator=gen)
    out = torch.empty_like(wide)
    y, z = pair(op, x, prec)
    lim = tol(sum(b.nterms for b in bs), z)

    def same(r):
        torch.cuda.synchronize()
        assert float((r - z).abs().max()) <= lim
        r.fill_(float("nan"))

    same(y)
    r = torch.full_like(x, float("nan"))
    for _ in range(3):
        op.apply_rows(wide, out, prec)
        op.apply_graph(x, r, prec)
        same(r)
    s = torch.cuda.Stream()
    E._capi.check(E.lib().sg4_plan_set_stream(op._h, C.c_void_p(s.cuda_stream)))
    torch.cuda.synchronize()
    op.apply_rows(x, r, prec)
    same(r)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        op.apply_rows(x, r, prec)
    for _ in range(3):
        op.apply_rows(wide, out, prec)
        torch.cuda.synchronize()
        graph.replay()
        same(r)
    xc = x.t().contiguous()
    rc = torch.empty_like(xc)
    op.apply(xc, rc, prec)
    rc.fill_(float("nan"))
    torch.cuda.synchronize()
    E._capi.check(E.lib().sg4_apply_noalloc(op._h, 4, C.c_void_p(xc.data_ptr()), C.c_void_p(rc.data_ptr()), prec))
    torch.cuda.synchronize()
    assert float((rc.t() - z).abs().max()) <= lim


@pytest.mark.parametrize("prec", [E.PREC_F32, E.PREC_F32X2])
def test_weight_indices_apart_from_the_places(prec):
    """A batch whose places and distinct term weights do not fit 32 bits
    together: the weight indices are kept beside the places."""
    bs = [E.SG4Basis(D, L) for D, L in [(12, 8), (11, 4), (10, 4), (9, 4), (8, 4), (7, 4), (6, 4), (5, 5), (4, 6)]]
    weights = {float(w) for b in bs for w in b.weights()}
    assert (len(weights) - 1).bit_length() + sum(b.sum_nb for b in bs).bit_length() > 32
    op = E.SG4Batch(bs, max_nvec=2)
    op.set_sparse(False)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(op.nb_ba, 2, device="cuda", dtype=torch.float64, generator=g)
    y, z = pair(op, x, prec)
    assert float((y - z).abs().max()) <= tol(max(b.nterms for b in bs), z)


def test_first_call_a_graph_and_noalloc_of_an_early_width():
    """A plan's first call may be its graph entry, and the allocation-free entry
    takes a width that was applied before the row sums were there."""
    b = E.SG4Basis(6, 6)
    g = torch.Generator(device="cuda").manual_seed(11)
    x = torch.randn(b.nb_ba, 8, device="cuda", dtype=torch.float64, generator=g)
    for prec in (E.PREC_FP64, E.PREC_F32, E.PREC_F32X2):
        first = E.SG4Operator(b, max_nvec=16)
        first.set_sparse(False)
        r = torch.full_like(x, float("nan"))
        for _ in range(3):
            first.apply_graph(x, r, prec)
        op = E.SG4Operator(b, max_nvec=16)
        op.set_sparse(False)
        xc = x.t().contiguous()
        rc = torch.empty_like(xc)
        op.apply(xc, rc, prec)                       # eight vectors: with atomics
        wide = torch.randn(b.nb_ba, 16, device="cuda", dtype=torch.float64, generator=g)
        y, z = pair(op, wide, prec)
        rc.fill_(float("nan"))
        torch.cuda.synchronize()
        E._capi.check(E.lib().sg4_apply_noalloc(op._h, 8, C.c_void_p(xc.data_ptr()), C.c_void_p(rc.data_ptr()), prec))
        y, z = pair(op, x, prec)
        assert float((r - z).abs().max()) <= tol(b.nterms, z), prec
        assert float((rc.t() - z).abs().max()) <= tol(b.nterms, z), prec
