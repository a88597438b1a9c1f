"""A two-mode function on the Smolyak set as one sparse matrix: the combination
weights over the levels of the other modes telescope to the two-mode
combination technique,

    <r|V_ab|r'> = sum_{l_a+l_b=m} M_ab(l_a,l_b) - sum_{l_a+l_b=m-1} M_ab(l_a,l_b),

m = L - (levels of the other modes' indices), M_ab the term's matrix of the
function.  Checked in numpy against the oracle's term-by-term sum, also with a
basis level below the grid level; one level off fails."""
import numpy as np
import pytest

from oracle import oracle as O


def pair_matrix(o, f, a, b, shift=0):
    D, L = o.D, int(np.max(o.lev.sum(1)))
    b1 = [[o.basis1d(k, l) for l in range(o.L + 1)] for k in range(D)]
    lam = [np.array([next(l for l in range(o.L + 1) if b1[k][l]["nb"] > i) for i in range(b1[k][-1]["nb"])])
           for k in range(D)]
    rows = {tuple(r): n for n, r in enumerate(o.packed)}
    M = {}

    def elem(la, lb, ia, ib, ja, jb):
        if la < 0 or lb < 0 or max(ia, ja) >= b1[a][la]["nb"] or max(ib, jb) >= b1[b][lb]["nb"]:
            return 0.0
        if (la, lb) not in M:
            A, B = b1[a][la], b1[b][lb]
            F = f(A["x"][:, None], B["x"][None, :])
            M[la, lb] = np.einsum("qi,q,qj,qs,sk,s,sl->ikjl", A["d0"], A["w"], A["d0"], F, B["d0"], B["w"], B["d0"],
                                  optimize=True)
        return M[la, lb][ia, ib, ja, jb]
    H = np.zeros((o.nb_ba, o.nb_ba))
    for n, r in enumerate(o.packed):
        m = L + shift - sum(lam[k][r[k]] for k in range(D) if k not in (a, b))
        for ja in range(len(lam[a])):
            for jb in range(len(lam[b])):
                c = list(r)
                c[a], c[b] = ja, jb
                n2 = rows.get(tuple(c))
                if n2 is not None:
                    H[n, n2] = sum(elem(la, s - la, r[a], r[b], ja, jb) * sg
                                   for s, sg in ((m, 1.0), (m - 1, -1.0)) for la in range(s + 1) if s <= o.L)
    return H


@pytest.mark.parametrize("D,L,LB,a,b", [(2, 4, 4, 0, 1), (3, 4, 4, 0, 2), (4, 3, 3, 1, 2), (3, 4, 2, 0, 1)])
def test_pair_telescoping_matches_smolyak_sum(D, L, LB, a, b):
    o = O.SG4(D, L, LB=LB)
    f = lambda x, y: np.exp(0.3 * x) * np.cos(0.7 * y) + x * y
    q = np.concatenate([o.term_grid(t) for t in range(o.nterms)])
    psi = np.random.default_rng(D).standard_normal((o.nb_ba, 2))
    ref = o.hpsi(psi, f(q[:, a], q[:, b]), np.zeros(D))
    got = pair_matrix(o, f, a, b) @ psi
    assert np.max(np.abs(got - ref)) < 1e-12 * np.max(np.abs(ref))
    assert np.max(np.abs(pair_matrix(o, f, a, b, -1) @ psi - ref)) > 1e-3 * np.max(np.abs(ref))
