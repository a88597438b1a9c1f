"""Applies of plans with so many packed rows that a thread per row and lane would
exceed the 2^32 threads of a launch."""
from host_hip import run

CODE = """
b = E.SG4Basis(3, 3)
t = E._capi.Tables()
C.memmove(C.byref(t), C.byref(b.tables), C.sizeof(t))
t.nb_ba = (1 << 28) + 1000          # rows that no term holds
h = C.c_void_p()
assert E.lib().sg4_plan_create(C.byref(t), 16, C.byref(h)) == 0
V, ck = np.ones(b.sum_nq), -0.5 * np.ones(3)
o = E._capi.Operator()
o.type_op, o.V, o.ck = 1, V.ctypes.data_as(E._capi.D_P), ck.ctypes.data_as(E._capi.D_P)
assert E.lib().sg4_plan_set_operator(h, C.byref(o)) == 0
x, y = C.c_void_p(1 << 40), C.c_void_p(1 << 44)
for nvec in (1, 3, 8, 16):
    for prec in (0, 1, 2):
        hh.hh_clear()
        assert E.lib().sg4_apply_rows(h, nvec, x, y, prec) == 0, (nvec, prec, E.lib().sg4_last_error())
        k = [l for l in log() if l[0] == "launch" and "spmm" in l[1]]
        assert len(k) == 1
        # the blocks reach the last row whatever the lanes per row
        assert int(k[0][2]) * int(k[0][4]) * 256 >= t.nb_ba or "any" in k[0][1]
"""


def test_rows_beyond_the_threads_of_a_launch():
    run(CODE)
