"""When a plan inverts its map for the row sums: not in applies that together
save less than it costs, and without the rows passing through the host."""
import pytest

from host_hip import run

CODE = """
hh.hh_fill(1)
b = E.SG4Basis(6, 6)          # 94 k places: ~0.6 ms against ~10 us an apply
op = E.SG4Operator(b, 16)
x, y = dev(16 * b.nb_ba), dev(16 * b.nb_ba)
at = None
for i in range(200):
    hh.hh_clear()
    assert E.lib().sg4_apply_rows(op._h, {nvec}, x, y, {prec}) == 0
    if launched("k_rs_fill"):
        at = i + 1
        assert launched("_out") == 1
        big = [l for l in log() if l[0] == "memcpyasync" and int(l[1]) >= 4 * b.nb_ba]
        assert not big, big
        break
    assert not launched("k_rs_")
assert at and 20 <= at <= 120, at
hh.hh_clear()
assert E.lib().sg4_apply_rows(op._h, {nvec}, x, y, {prec}) == 0
assert not launched("k_rs_fill") and launched("_out") == 1
"""


@pytest.mark.parametrize("nvec,prec", [(1, 0), (16, 0), (3, 1), (8, 2)])
def test_the_map_is_inverted_when_it_has_paid(nvec, prec):
    run(CODE.format(nvec=nvec, prec=prec))
