"""Setting an operator when the device is short of memory: the sparse-matrix
tables and workspaces are not needed (the kinetic matrix then comes from the host,
FP64 takes the term kernels), what is needed is reported as such."""
import pytest

from host_hip import run

CODE = """
hh.hh_fill(0)
b = E.SG4Basis(3, 3)
V, ck = np.ones(b.sum_nq), -0.5 * np.ones(3)
o = E._capi.Operator()
o.type_op, o.V, o.ck = 1, V.ctypes.data_as(E._capi.D_P), ck.ctypes.data_as(E._capi.D_P)
x, y = dev(b.nb_ba), dev(b.nb_ba)
h = C.c_void_p()
assert E.lib().sg4_plan_create(C.byref(b.tables), 4, C.byref(h)) == 0
hh.hh_clear()
assert E.lib().sg4_plan_set_operator(h, C.byref(o)) == 0
total = sum(l[0] == "malloc" for l in log())
assert total > 10
ok = 0
for n in range(total):
    h = C.c_void_p()
    assert E.lib().sg4_plan_create(C.byref(b.tables), 4, C.byref(h)) == 0
    hh.hh_clear()
    hh.hh_allow(n)                     # the n-th allocation from here fails
    rc = E.lib().sg4_plan_set_operator(h, C.byref(o))
    hh.hh_allow(-1)
    assert any(l[0] == "nomem" for l in log())
    assert rc in (E._capi.OK, E._capi.ERR_OOM), (n, rc)
    if rc == E._capi.OK:
        ok += 1
        sp, nnz = C.c_int32(), C.c_int64()
        assert E.lib().sg4_plan_split_info(h, C.byref(sp), C.byref(nnz)) == 0 and sp.value == 1
        for prec in (0, 1, 2):
            assert E.lib().sg4_apply_rows(h, 1, x, y, prec) == 0
        assert E.lib().sg4_plan_set_operator(h, C.byref(o)) == 0
    assert E.lib().sg4_plan_destroy(h) == 0
assert ok >= total - 2, (ok, total)    # the coefficients and the terms themselves
"""


def test_one_failed_allocation_in_the_set_up():
    run(CODE)
