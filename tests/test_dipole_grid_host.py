"""sg4_cheby_field_gradient takes a dipole operator with the rows of H; mu has a
value per grid point of H.  The comparison of the dipole operator's potential
with mu is made only between equal grids: another plan's grid may be larger than
mu (here 129 points against 63, 25 rows both)."""
import pytest

from host_hip import run

CODE = """
hh.hh_fill(0)
b = E.SG4Basis(2, 3, 3)
H = E.SG4Operator(b, 4)
c = E.SG4Basis(2, {L}, 3)
assert c.nb_ba == b.nb_ba and (c.sum_nq == b.sum_nq) == ({L} == 3)
Mu = E.SG4Operator(c, 4, potential=np.zeros(c.sum_nq), ck=np.zeros(2))
{before}
eps, coef = np.full(8, 0.1), np.ones(6)
p = E._capi.ChebyParams()
p.dt, p.Esc, p.ncoef, p.nseg, p.steps_per_seg, p.ckpt_every = 0.1, 1.0, 6, 8, 1, 2
p.coef, p.eps = coef.ctypes.data_as(E._capi.D_P), eps.ctypes.data_as(E._capi.D_P)
rows = (C.c_int64 * 2)(0, b.nb_ba)
J, g = C.c_double(), np.zeros(8)
hh.hh_clear()
rc = E.lib().sg4_cheby_field_gradient(H._h, Mu._h, dev(b.sum_nq), 1, dev(2 * b.nb_ba), dev(2 * b.nb_ba), 1, rows,
                                      C.byref(p), C.byref(J), g.ctypes.data_as(E._capi.D_P))
assert rc == 0
assert launched("k_differ") == {compared}, launched("k_differ")
assert (launched("k_nm_order") > 0) == {matrix}
"""


@pytest.mark.parametrize("L,before,compared,matrix", [
    (3, "", 1, True), (4, "", 0, False), (3, "Mu.set_sparse(False)", 0, False),
    (3, "Mu.set_deterministic(True)", 0, False)])
def test_only_equal_grids_are_compared(L, before, compared, matrix):
    run(CODE.format(L=L, before=before, compared=compared, matrix=matrix))
