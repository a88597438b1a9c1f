"""sg4_plan_config reports the launch that the next apply takes: the plain one
while the terms add with atomics, the one derived from the sizes once their
results are summed row by row."""
import pytest

from host_hip import run

CODE = """
PLAIN = dict(nthreads=256, lds_budget=65536, grid=0, xcd=0)
small = E.SG4Operator(E.SG4Basis(4, 4), 4)
assert small.config(2, {prec}) == PLAIN          # below the places that are summed row by row
hh.hh_fill(1)
b = E.SG4Basis(6, 6)
op = E.SG4Operator(b, 16)
x, y = dev(16 * b.nb_ba), dev(16 * b.nb_ba)
def kernel(w):
    hh.hh_clear()
    assert E.lib().sg4_apply_rows(op._h, w, x, y, {prec}) == 0
    return [l for l in log() if l[0] == "launch" and ("k_hpsi" in l[1])][-1]
assert op.config(2, {prec}) == PLAIN and int(kernel(2)[5]) == 256
assert op.config(2, {prec}) == PLAIN
assert E.lib().sg4_apply_graph(op._h, 1, x, y, {prec}) == 0      # inverts the map
c = op.config(2, {prec})
assert c["lds_budget"] < 65536 and "_out" in kernel(2)[1]
assert c["nthreads"] == max(256, int(kernel(2)[5]))
op.set_deterministic(True)
assert op.config(2, {prec}) == PLAIN and "_out" not in kernel(2)[1]
op.set_deterministic(False)
hh.hh_limit(hh.hh_held() + (3 << 20))     # lists fit, 16 columns of results do not
assert "_out" not in kernel(16)[1] and op.config(16, {prec}) == PLAIN
assert op.config(2, {prec}) == c
op.set_config(2, {prec}, 512, 40960, 0, 3)
assert op.config(2, {prec}) == dict(nthreads=512, lds_budget=40960, grid=0, xcd=3)
"""


@pytest.mark.parametrize("prec", [0, 1, 2])
def test_config_is_the_launch_in_use(prec):
    run(CODE.format(prec=prec))
