"""The autotuner switches the sparse matrix and the timing off for its launches;
both are as before after it ended with an error of the runtime."""
import pytest

from host_hip import run

CODE = """
hh.hh_fill(0)
op = E.SG4Operator(E.SG4Basis(3, 3), 4)
assert op.sparse_info()[0]
op.timing(True)
x, y = dev(200), dev(200)
hh.hh_fail_record({n})
ms = C.c_float()
assert E.lib().sg4_plan_autotune(op._h, 1, 0, C.byref(ms)) == E._capi.ERR_HIP
hh.hh_fail_record(0)
assert op.sparse_info()[0]
hh.hh_clear()
assert E.lib().sg4_apply_rows(op._h, 1, x, y, 0) == 0
assert launched("spmm") == 1 and not launched("k_hpsi")
assert len(op.kernel_times()) == 1
"""


@pytest.mark.parametrize("n", [1, 2, 7])
def test_an_error_in_the_autotuner_leaves_the_plan_as_it_was(n):
    run(CODE.format(n=n))
