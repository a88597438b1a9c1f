"""Kernel times and statistics of a propagation: one record per H.psi, with the
vectors of its applies, on the sparse matrix as by the term kernels."""
from host_hip import run

CODE = """
hh.hh_fill(0)
b = E.SG4Basis(2, 3, 3)
H, Mu = E.SG4Operator(b, 4), E.SG4Operator(b, 4, potential=np.zeros(b.sum_nq), ck=np.zeros(2))
eps, coef = np.full(8, 0.1), np.ones(6)
p, t = E._capi.ChebyParams(), E._capi.TaylorParams()
p.dt, p.Esc, p.ncoef, p.nseg, p.steps_per_seg, p.ckpt_every = 0.1, 1.0, 6, 8, 1, 8
t.dt, t.npoly, t.poly_tol, t.nseg, t.steps_per_seg = 0.1, 3, 1e-20, 8, 1
p.coef = coef.ctypes.data_as(E._capi.D_P)
p.eps = t.eps = eps.ctypes.data_as(E._capi.D_P)
rows = (C.c_int64 * 2)(0, b.nb_ba)
J, g = C.c_double(), np.zeros(8)
mu, x, y = dev(b.sum_nq), dev(2 * b.nb_ba), dev(2 * b.nb_ba)
got = []
for sparse in (True, False):
    H.set_sparse(sparse)
    for call in (lambda: E.lib().sg4_cheby_propagate(H._h, mu, 1, x, C.byref(p)),
                 lambda: E.lib().sg4_cheby_field_gradient(H._h, Mu._h, mu, 1, x, y, 1, rows, C.byref(p), C.byref(J),
                                                          g.ctypes.data_as(E._capi.D_P)),
                 lambda: E.lib().sg4_taylor_propagate(H._h, mu, 1, x, C.byref(t), None)):
        hh.hh_clear()
        H.timing(True)
        assert call() == 0
        got.append((sparse, len(H.kernel_times()), H.stats(2)["flops"]))
        H.timing(False)
        assert (launched("k_nm_order") + launched("spmm") > 0 and launched("k_hpsi") == 0) == sparse
assert [r[1:] for r in got[:3]] == [r[1:] for r in got[3:]], got
assert got[0][1] == 8 * 5 and got[0][2] > 0
"""


def test_records_of_a_propagation_do_not_depend_on_the_route():
    run(CODE)
