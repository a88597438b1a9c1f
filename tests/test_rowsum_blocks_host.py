"""The blocks that hold the terms' results: kept when a wider one does not fit
the device memory, given back with the plan's graphs and after an autotuner run
that leaves them without a use.  (Fresh memory of ones: the row check fails, so
FP64 takes the term kernels, and the inverted map comes out non-empty.)"""
import pytest

from host_hip import run

PLAN = """
hh.hh_fill(1)
b = E.SG4Basis(6, 6)
assert b.sum_nb >= 1 << 16
op = E.SG4Operator(b, 32)
assert not op.sparse_info()[0]
x, y, u, v = dev(32 * b.nb_ba), dev(32 * b.nb_ba), dev(32 * b.nb_ba), dev(32 * b.nb_ba)
block = lambda w: 8 * b.sum_nb * w + 255 & ~255
def rows(w):
    hh.hh_clear()
    assert E.lib().sg4_apply_rows(op._h, w, x, y, 0) == 0
    return "sums" if launched("k_hpsi_t1s_out_f64") else "atomics" if launched("k_hpsi_t1s_f64") else None
def graph(w):
    assert E.lib().sg4_apply_graph(op._h, w, u, v, 0) == 0
def tries(n):
    return [l[0] for l in log() if l[0] in ("malloc", "nomem") and int(l[1]) == n]
graph(1)                                  # builds the inverted map
assert rows(2) == "sums" and tries(block(2)) == ["malloc"]
"""


def test_a_block_that_does_not_fit_leaves_the_smaller_one():
    run(PLAN + """
assert rows(4) == "sums" and rows(2) == "sums"
hh.hh_limit(hh.hh_held() + block(8))      # 8 columns fit, 16 do not
assert rows(8) == "sums"
assert rows(16) == "atomics" and tries(block(16)) == ["nomem"]
for i in range(4):                        # neither width allocates again
    assert rows(8) == "sums" and not tries(block(8))
    assert rows(16) == "atomics" and not tries(block(16))
    assert rows(32) == "atomics" and not tries(block(32))
""")


def test_graphs_of_growing_widths_hold_one_block():
    run(PLAN + """
held = hh.hh_held()
for w in range(2, 12):
    graph(w)
assert rows(24) == "sums" and rows(3) == "sums"
# ten widths would be 65 columns of results; one block of 11 stays
assert hh.hh_held() - held < block(11) + block(24) + (16 << 20), (hh.hh_held() - held, block(1))
hh.hh_clear()
op.set_config(1, E.PREC_FP64)             # drops the graphs
freed = [int(l[1]) for l in log() if l[0] == "free"]
assert block(11) in freed, freed
""")


def test_graphs_leave_room_for_other_streams():
    run(PLAN + """
for w in range(2, 12):
    graph(w)
for stream in (0x7000, 0x7010):
    assert E.lib().sg4_plan_set_stream(op._h, C.c_void_p(stream)) == 0
    assert rows(12) == "sums" and rows(3) == "sums"
""")


# zeros: rows and grid pass the checks, and H is a matrix without entries
def test_autotuning_the_term_kernels_of_a_matrix_leaves_no_block():
    run("""
hh.hh_fill(0)
b = E.SG4Basis(6, 6)
op = E.SG4Operator(b, 4)
assert op.sparse_info()[0]
hh.hh_fill(1)
hh.hh_clear()
op.autotune(4)
n = 8 * b.sum_nb * 4 + 255 & ~255
made = [l[2] for l in log() if l[0] == "malloc" and int(l[1]) == n]
gone = [l[2] for l in log() if l[0] == "free" and int(l[1]) == n]
assert made and sorted(made) == sorted(gone), (made, gone)
""")
