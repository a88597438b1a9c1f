"""Setting an operator leaves no work in flight on the plan's stream: a caller
may hand the plan another stream next, which does not wait for the first."""
import pytest

from host_hip import run

CODE = """
hh.hh_fill({fill})
b = E.SG4Basis(3, 3)
op = E.SG4Operator(b, 4)
V = np.ones(b.sum_nq)
ck = -0.5 * np.ones(3)
o = E._capi.Operator()
o.type_op, o.V, o.ck = 1, V.ctypes.data_as(E._capi.D_P), ck.ctypes.data_as(E._capi.D_P)
def idle():
    last = max((i for i, l in enumerate(log()) if l[0] in ("launch", "memcpyasync")), default=-1)
    assert any(l[0] == "sync" for l in log()[last + 1:]), log()[-4:]
for call in (lambda: E.lib().sg4_plan_set_operator(op._h, C.byref(o)),
             lambda: E.lib().sg4_plan_set_option(op._h, E._capi.OPT_GROUPING, 1),
             lambda: E.lib().sg4_plan_set_henon_heiles(op._h, 0.1)):
    hh.hh_clear()
    assert call() == 0
    idle()
"""


# fresh memory of zeros: rows and grid pass the checks (kinetic and whole
# matrix are built); of ones: they do not (the kinetic matrix comes from the host)
@pytest.mark.parametrize("fill", [0, 1])
def test_set_operator_returns_with_its_matrices_written(fill):
    run(CODE.format(fill=fill))
