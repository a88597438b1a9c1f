"""Work that users of the SG4 H.psi library have it do, for timing it.

Each case goes through a public entry point: block applies of H.psi in the
three precision modes (`SG4Operator.apply`, what a Davidson or a propagation
driver calls), the type-10 and general type-1 operators, the grid gradient
(`SG4Operator.grad_V`), the device propagator and its adjoint gradient
(`propagate_device`, `field_gradient_device`) and the dense block products of
the Davidson (`sg4_block_gram`, `sg4_block_combine`).

Operators: the Henon-Heiles model of the library's tests ("hh"), evaluated on
the device, and a potential energy surface given as grid values that couples
all modes ("pes"), which is what a host program with its own potential hands
over.  The parameters of both are drawn from the seed.
"""
import ctypes as C
import math

import numpy as np
import torch

import elvibrot_amd as E
from elvibrot_amd import potentials
from elvibrot_amd.propagation import ChebyshevPropagator, field_gradient_device, propagate_device

DEV = "cuda:0"
PREC = {"fp64": E.PREC_FP64, "f32": E.PREC_F32, "f32x2": E.PREC_F32X2}
# the launches that the benchmark of the 10D L=8 block-16 workload sets
BENCH_LAUNCH = {"fp64": (512, 163840, 2048, 3), "f32x2": (1024, 163840, 512, 2)}


def listed():
    return [
        # one packed vector of the reference's 6D test: the smallest apply, all latency
        dict(name="hpsi 6D L3 x1", kind="hpsi", D=6, L=3, nvec=1, prec="fp64", pot="hh", launch="default"),
        # a Davidson block of the 6D L=6 model
        dict(name="hpsi 6D L6 x16", kind="hpsi", D=6, L=6, nvec=16, prec="fp64", pot="hh", launch="default"),
        # the headline workload, FP64 and split precision, with the benchmark's launches
        dict(name="hpsi 10D L8 x16", kind="hpsi", D=10, L=8, nvec=16, prec="fp64", pot="hh", launch="bench"),
        dict(name="hpsi 10D L8 x16 split", kind="hpsi", D=10, L=8, nvec=16, prec="f32x2", pot="hh", launch="bench"),
        # an odd block on a potential that couples all modes, as a host program's surface does
        dict(name="hpsi 9D L7 x5 pes", kind="hpsi", D=9, L=7, nvec=5, prec="fp64", pot="pes", launch="default"),
        # the FP32 mode on a wide block
        dict(name="hpsi 8D L6 x24 f32 pes", kind="hpsi", D=8, L=6, nvec=24, prec="f32", pot="pes", launch="default"),
        # the curvilinear (type 10) operator of the triatomic, the block of its 5 lowest levels
        dict(name="jacobi L10 x5", kind="jacobi", L=10, nvec=5),
        # position-dependent coefficients with first, second and mixed derivatives
        dict(name="type1 5D L5 x4", kind="type1", D=5, L=5, nvec=4),
        # Hellmann-Feynman gradients of a block of eigenvectors on all grid points
        dict(name="grad 8D L6 x5", kind="grad", D=8, L=6, nvec=5, pot="hh"),
        # one complex state in each of a batch of uneven instances under a field
        dict(name="field 12 instances", kind="field", ninst=12, Dlo=4, Dhi=9, Llo=4, Lhi=6, nseg=3, steps=2),
        # the gradient of the final overlaps with respect to the field
        dict(name="field gradient 3 instances", kind="fieldgrad", ninst=3, Dlo=3, Dhi=5, Llo=4, Lhi=5, nseg=3, steps=2),
        # the dense products of a Davidson iteration over 10D L=8 vectors: new columns of the
        # projected matrix and the wanted Ritz vectors
        dict(name="subspace 10D L8", kind="subspace", n=1256465, m=60, q=16, k=20, d=60),
    ]


def draw(rng):
    kind = rng.choices(["hpsi", "jacobi", "type1", "grad", "field", "fieldgrad", "subspace"],
                       [8, 1, 1, 1, 1, 1, 1])[0]
    logint = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))
    if kind == "hpsi":
        while True:
            c = dict(kind=kind, D=rng.randint(2, 12), L=rng.randint(2, 8), nvec=logint(1, 40),
                     prec=rng.choices(["fp64", "f32", "f32x2"], [6, 1, 1])[0],
                     pot=rng.choice(["hh", "pes"]), launch="default")
            n = _sum_n(c["D"], c["L"])
            # the surface's grid values are made on the host: fewer points
            if 300 <= n <= (8e6 if c["pot"] == "pes" else 3.2e7) and n * c["nvec"] <= 5e8:
                return c
    if kind == "jacobi":
        return dict(kind=kind, L=rng.randint(4, 12), nvec=logint(1, 24))
    if kind == "type1":
        return dict(kind=kind, D=rng.randint(2, 6), L=rng.randint(3, 6), nvec=logint(1, 16))
    if kind == "grad":
        return dict(kind=kind, D=rng.randint(3, 8), L=rng.randint(3, 6), nvec=logint(1, 16),
                    pot=rng.choice(["hh", "pes"]))
    if kind == "field":
        return dict(kind=kind, ninst=logint(1, 12), Dlo=3, Dhi=rng.randint(4, 9), Llo=4,
                    Lhi=rng.randint(4, 6), nseg=rng.randint(1, 3), steps=rng.randint(1, 2))
    if kind == "fieldgrad":
        return dict(kind=kind, ninst=logint(1, 4), Dlo=2, Dhi=rng.randint(3, 5), Llo=3,
                    Lhi=rng.randint(4, 5), nseg=rng.randint(2, 3), steps=rng.randint(1, 2))
    m = rng.randint(1, 84)
    return dict(kind="subspace", n=logint(5000, 1250000), m=m, q=rng.randint(1, 20), k=rng.randint(1, 24), d=m)


# ---- what a user's program has in hand ----------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _block(nvec, nb, seed):
    """A block of normalised packed vectors, column-major (nvec, nb)."""
    x = torch.randn(nvec, nb, device=DEV, dtype=torch.float64, generator=_gen(seed))
    return x / torch.linalg.norm(x, dim=1, keepdim=True)


def _lam(seed):
    return 0.111803 * (0.8 + 0.4 * np.random.default_rng(seed).random())


def _pes(D, seed):
    """V(q) of a surface that couples all modes: harmonic and cubic parts and a
    Gaussian barrier in all coordinates."""
    r = np.random.default_rng(seed)
    w = torch.tensor(0.8 + 0.4 * r.random(D), device=DEV)
    c = torch.tensor(0.1 * r.standard_normal((D, D)), device=DEV)
    a, b = 0.5 + 0.5 * r.random(), 0.1 + 0.1 * r.random()

    def V(q):
        s = q * q
        return 0.5 * s @ w + ((s @ c) * q).sum(1) / D + a * torch.exp(-b * s.sum(1))
    return V


def _operator(c, seed, max_nvec):
    b = E.SG4Basis(c["D"], c["L"])
    if c["pot"] == "hh":
        return E.SG4Operator(b, max_nvec=max_nvec, potential=("henon_heiles", _lam(seed)))
    V = _Sparse(c["D"], c["L"]).on_grid(_pes(c["D"], seed)).cpu().numpy()
    return E.SG4Operator(b, max_nvec=max_nvec, potential=V, ck=-0.5 * np.ones(c["D"]))


def _type1_terms(D, seed):
    """Derivative terms and coefficient functions of a general type-1 operator:
    V - 1/2 sum_k g_k(q) d_k^2, first derivatives, and a mixed derivative."""
    r = np.random.default_rng(seed)
    V = _pes(D, seed)
    amp = 0.1 + 0.1 * r.random(D)
    der, fun = [(-1, -1)], [V]
    for k in range(D):
        der.append((k, k))
        fun.append(lambda q, k=k: -0.5 / (1.0 + amp[k] * q[:, (k + 1) % D] ** 2))
    for k in range(D):
        der.append((k, -1))
        fun.append(lambda q, k=k: 0.05 * torch.sin(q[:, k]))
    if D > 1:
        der.append((0, 1))
        fun.append(lambda q: 0.1 * torch.cos(q[:, 0] + q[:, 1]))
    return der, fun


def _instances(c):
    """The uneven instances of a batch (D, L), the same for every seed."""
    r = np.random.default_rng(7)
    D = r.integers(c["Dlo"], c["Dhi"] + 1, size=c["ninst"])
    L = r.integers(c["Llo"], c["Lhi"] + 1, size=c["ninst"])
    return [(int(d), int(l)) for d, l in zip(D, L)]


def _field(c, seed):
    return np.random.default_rng(seed).normal(0.0, 0.05, c["nseg"])


# dt of a Chebyshev step, and a spectral range that holds what spectral_bounds
# gives for these operators (3D L=4: 1.1..10.4, 4D L=6: 1.3..16.9, 9D L=4:
# 4.1..13.4, 9D L=6: 3.8..19.4) and the field
DT = 0.1


def _range(insts):
    return 0.0, max(3.0 * l + 0.5 * d for d, l in insts)


def prepare(case, seed):
    c = case
    if c["kind"] in ("hpsi", "jacobi", "type1"):
        mx = max(16, c["nvec"])
        if c["kind"] == "hpsi":
            op = _operator(c, seed, mx)
            if c["launch"] == "bench":
                op.set_config(c["nvec"], PREC[c["prec"]], *BENCH_LAUNCH[c["prec"]])
        elif c["kind"] == "jacobi":
            r = np.random.default_rng(seed)
            op = potentials.jacobi_triatomic_operator(c["L"], max_nvec=mx, coupling=0.005 + 0.01 * r.random())
        else:
            b = E.SG4Basis(c["D"], c["L"])
            der, fun = _type1_terms(c["D"], seed)
            S = _Sparse(c["D"], c["L"])
            F = torch.stack([S.on_grid(f) for f in fun]).cpu().numpy()
            op = E.SG4Operator(b, max_nvec=mx, potential=("type1", der, F))
        x = _block(c["nvec"], op.nb_ba, seed)
        return dict(kind="apply", op=op, x=x, y=torch.empty_like(x), prec=PREC[c.get("prec", "fp64")])
    if c["kind"] == "grad":
        op = _operator(c, seed, max(16, c["nvec"]))
        x = _block(c["nvec"], op.nb_ba, seed).T.contiguous()
        return dict(kind="grad", op=op, x=x,
                    g=torch.empty(op.basis.sum_nq, c["nvec"], device=DEV, dtype=torch.float64))
    if c["kind"] in ("field", "fieldgrad"):
        insts = _instances(c)
        op = E.SG4Batch([E.SG4Basis(d, l) for d, l in insts], max_nvec=4,
                        potential=("henon_heiles", _lam(seed)))
        mu = op.grid_dipole()
        lo, hi = _range(insts)
        p = ChebyshevPropagator(op, DT, lo, hi, mu=mu)
        psi, target = _states(op.row0, seed)
        st = dict(kind=c["kind"], prop=p, psi=psi, eps=_field(c, seed), steps=c["steps"])
        if c["kind"] == "fieldgrad":
            st.update(target=target, blocks=list(zip(op.row0[:-1], op.row0[1:])))
            p.mu_s(psi * 0)          # the dipole operator's plan, kept with the propagator
        return st
    n, g = c["n"], _gen(seed)
    op = E.SG4Operator(E.SG4Basis(3, 2), max_nvec=4)      # gives the products their stream
    V = torch.randn(c["d"], n, device=DEV, dtype=torch.float64, generator=g) / math.sqrt(n)
    H = torch.randn(c["q"], n, device=DEV, dtype=torch.float64, generator=g) / math.sqrt(n)
    U = torch.randn(c["k"], c["d"], device=DEV, dtype=torch.float64, generator=g) / math.sqrt(c["d"])
    need = C.c_int64()
    E._capi.check(E.lib().sg4_block_gram_work(c["m"], c["q"], C.byref(need)))
    f64 = dict(device=DEV, dtype=torch.float64)
    return dict(kind="subspace", op=op, V=V, H=H, U=U, work=torch.empty(need.value, **f64),
                G=torch.empty(c["m"], c["q"], **f64), X=torch.empty(c["k"], n, **f64))


def _states(row0, seed):
    """One complex packet per instance (a few of the lowest rows) and a target."""
    nb = int(row0[-1])
    r = np.random.default_rng(seed)
    psi = np.zeros((1, nb), dtype=np.complex128)
    tgt = np.zeros((1, nb), dtype=np.complex128)
    for r0, r1 in zip(row0[:-1], row0[1:]):
        n = min(40, int(r1 - r0))
        for a in (psi, tgt):
            v = (r.standard_normal(n) + 1j * r.standard_normal(n)) * np.exp(-0.1 * np.arange(n))
            a[0, r0:r0 + n] = v / np.linalg.norm(v)
    return torch.tensor(psi, device=DEV), torch.tensor(tgt, device=DEV)


# ---- one pass -------------------------------------------------------------------
def run(state):
    s = state
    if s["kind"] == "apply":
        return s["op"].apply(s["x"], s["y"], s["prec"])
    if s["kind"] == "grad":
        return s["op"].grad_V(s["x"], s["x"], s["g"])
    if s["kind"] == "field":
        return propagate_device(s["prop"], s["psi"], s["eps"], s["steps"])
    if s["kind"] == "fieldgrad":
        J, g = field_gradient_device(s["prop"], s["psi"], s["target"], s["eps"], s["steps"],
                                     checkpoint_every=2, blocks=s["blocks"])
        return dict(J=J, grad=g)
    p, lib, chk = (lambda t: C.c_void_p(t.data_ptr())), E.lib(), E._capi.check
    V, H, U, G, X = s["V"], s["H"], s["U"], s["G"], s["X"]
    chk(lib.sg4_block_gram(s["op"]._h, G.shape[0], G.shape[1], V.shape[1], p(V), V.stride(0), p(H),
                           H.stride(0), p(G), p(s["work"]), s["work"].numel()))
    chk(lib.sg4_block_combine(s["op"]._h, U.shape[0], U.shape[1], V.shape[1], p(U), p(V), V.stride(0),
                              0.0, p(X), X.stride(0)))
    return G, X


# ---- sizes ----------------------------------------------------------------------
def _poly(D, L, f):
    """[z^s] (sum_l f(l) z^l)^D for s = 0..L"""
    g = [1.0] + [0.0] * L
    for _ in range(D):
        g = [sum(g[s - l] * f(l) for l in range(s + 1)) for s in range(L + 1)]
    return g


def _sum_n(D, L, f=lambda l: 1.0 + 2 * l):
    return sum(_poly(D, L, f)[max(0, L - D + 1):])


def _rows(D, L, band=lambda l: 1.0 if l == 0 else 2.0):
    return sum(_poly(D, L, band))


def _flops(D, L, f=lambda l: 1.0 + 2 * l):
    """Of one product of every term's values with the matrix of each of its modes
    (n_k > 1): sum_t sum_k 2 N_t n_k."""
    rest = _poly(D - 1, L, f)
    lo = max(0, L - D + 1)
    return sum(D * 2.0 * f(l) ** 2 * rest[s - l] for s in range(lo, L + 1) for l in range(s + 1) if f(l) > 1)


def work(case):
    c = case
    if c["kind"] == "subspace":
        n = c["n"]
        return dict(bytes=8.0 * n * (c["m"] + c["q"] + c["d"] + c["k"]) + 8.0 * (c["m"] * c["q"] + c["k"] * c["d"]),
                    flops=2.0 * n * (c["m"] * c["q"] + c["k"] * c["d"]))
    if c["kind"] in ("field", "fieldgrad"):
        insts = _instances(c)
        lo, hi = _range(insts)
        orders = 0.5 * (hi - lo) * DT + 12
        naps = orders * c["nseg"] * c["steps"] * (1 if c["kind"] == "field" else 5)
        # each order reads the state and the potential and writes the new state
        by = sum(32.0 * _rows(d, l) + 8.0 * _sum_n(d, l) for d, l in insts)
        fl = sum(2.0 * (2 * _flops(d, l) + _sum_n(d, l)) for d, l in insts)
        return dict(bytes=by * naps, flops=fl * naps)
    if c["kind"] == "jacobi":
        f = lambda l: 2.0 + 2 * l
        nb, nq = _rows(3, c["L"], lambda l: 2.0), _sum_n(3, c["L"], f)
        return dict(bytes=16.0 * nb * c["nvec"] + 96.0 * nq, flops=4 * _flops(3, c["L"], f) * c["nvec"])
    D, L, nv = c["D"], c["L"], c["nvec"]
    nb, nq = _rows(D, L), _sum_n(D, L)
    if c["kind"] == "grad":
        return dict(bytes=8.0 * nv * (nb + nq), flops=(_flops(D, L) + 2 * nq) * nv)
    if c["kind"] == "type1":
        nder = 2 * D + 1 + (D > 1)
        return dict(bytes=16.0 * nb * nv + 8.0 * nder * nq, flops=(4 * _flops(D, L) + 2 * nder * nq) * nv)
    return dict(bytes=16.0 * nb * nv + 8.0 * nq, flops=(2 * _flops(D, L) + nq) * nv)


# ---- the same in plain torch / numpy ----------------------------------------------
def _hermite(n, nb, x):
    """Orthonormal Hermite functions 0..nb-1 and two derivatives at x."""
    p = np.zeros((nb + 3, len(x)))
    p[0] = np.pi ** -0.25 * np.exp(-0.5 * x * x)
    p[1] = np.sqrt(2.0) * x * p[0]
    for k in range(2, nb + 3):
        p[k] = np.sqrt(2.0 / k) * x * p[k - 1] - np.sqrt((k - 1.0) / k) * p[k - 2]
    k = np.arange(nb)[:, None]
    low = np.concatenate([np.zeros((1, len(x))), p])[:nb]
    d1 = np.sqrt(k / 2.0) * low - np.sqrt((k + 1) / 2.0) * p[1:nb + 1]
    d2 = (x * x - 2 * k - 1) * p[:nb]
    return p[:nb].T, d1.T, d2.T


def _rule(kind, n, Q0, scale):
    """nodes, basis->grid, grid->basis, first and second grid derivatives (n points, n functions)"""
    if kind == "ho":
        x, _ = np.polynomial.hermite.hermgauss(n)
        d0, d1, d2 = _hermite(n, n, x)
        w = 1.0 / (d0 * d0).sum(1)
        s = math.sqrt(scale)
        q, d0, d1, d2, w = Q0 + x / scale, s * d0, s * scale * d1, s * scale ** 2 * d2, w / scale
    else:
        x, w = np.polynomial.legendre.leggauss(n)
        P = np.polynomial.legendre.legvander(x, n - 1)
        nrm = np.sqrt(np.arange(n) + 0.5)
        dP = np.stack([np.polynomial.legendre.legval(x, np.polynomial.legendre.legder(np.eye(n)[j])) for j in range(n)], 1)
        sn = np.sqrt(1 - x * x)
        d0, d1 = P * nrm, -sn[:, None] * dP * nrm
        ll = np.arange(n) * (np.arange(n) + 1.0)
        d2 = (-(x / sn)[:, None] * (-sn[:, None] * dP) - ll * P) * nrm
        q = np.arccos(x)
    inv = np.linalg.inv(d0)
    t = lambda a: torch.tensor(np.ascontiguousarray(a), device=DEV)
    return dict(q=t(q), wq=t(w), B=t(d0), Bt=t((d0 * w[:, None]).T), D1=t(d1 @ inv), D2=t(d2 @ inv))


class _Sparse:
    """The Smolyak terms and packed rows of D modes at level L, nA + nB l
    functions and points per mode; terms with equal sizes handled together."""

    def __init__(self, D, L, modes=None, nA=1, nB=2):
        self.D, self.L = D, L
        n = [nA + nB * l for l in range(L + 1)]
        modes = modes or [("ho", 0.0, 1.0)] * D
        same = len(set(modes)) == 1
        self.mode_id = [0] * D if same else list(range(D))
        self.rules = {(i, l): _rule(modes[i][0], n[l], modes[i][1], modes[i][2])
                      for i in set(self.mode_id) for l in range(L + 1)}
        self.n = np.array(n)
        # levels, the first mode's fastest
        lev, left = np.zeros((1, 0), dtype=np.int64), np.array([L])
        for _ in range(D):
            rep = left + 1
            l = np.arange(rep.sum()) - np.repeat(np.cumsum(rep) - rep, rep)
            lev, left = np.hstack([l[:, None], np.repeat(lev, rep, 0)]), np.repeat(left, rep) - l
        keep = L - left >= max(0, L - D + 1)
        self.lev, left = lev[keep], left[keep]
        self.wgt = np.array([(-1.0) ** j * math.comb(D - 1, int(j)) for j in left])
        self.nt = self.n[self.lev].prod(1)
        self.off = np.concatenate([[0], np.cumsum(self.nt)])
        # packed rows, the last mode's index fastest; level of a 1-D index
        lam = np.searchsorted(self.n, np.arange(n[-1]), side="right")
        self.cnt = [int((lam <= r).sum()) for r in range(L + 1)]
        code, left = np.zeros(1, dtype=np.int64), np.array([L])
        for _ in range(D):
            rep = np.array(self.cnt)[left]
            i = np.arange(rep.sum()) - np.repeat(np.cumsum(rep) - rep, rep)
            code, left = np.repeat(code, rep) * (n[-1] + 1) + i, np.repeat(left, rep) - lam[i]
        self.code, self.base = torch.tensor(code, device=DEV), n[-1] + 1
        self.nb = len(code)
        groups = {}
        key = [tuple((self.mode_id[k], int(l)) for k, l in enumerate(t) if l or nA > 1) for t in self.lev]
        for t, k in enumerate(key):
            groups.setdefault(k, []).append(t)
        self.groups = [(k, np.array(ts)) for k, ts in groups.items()]

    def chunks(self, points):
        for k, ts in self.groups:
            per = max(1, int(points // self.nt[ts[0]]))
            for a in range(0, len(ts), per):
                yield k, ts[a:a + per]

    def digits(self, ts):
        """0-based mode indices of every point of the terms ts: (T, N, D)"""
        nk = torch.tensor(self.n[self.lev[ts]], device=DEV)
        p = torch.arange(int(self.nt[ts[0]]), device=DEV)[None, :].expand(len(ts), -1)
        out = []
        for k in range(self.D):
            out.append(p % nk[:, k:k + 1])
            p = p // nk[:, k:k + 1]
        return torch.stack(out, 2)

    def rows(self, ts):
        d = self.digits(ts)
        code = torch.zeros_like(d[:, :, 0])
        for k in range(self.D):
            code = code * self.base + d[:, :, k]
        return torch.searchsorted(self.code, code)

    def points(self, ts):
        """coordinates (T, N, D)"""
        d = self.digits(ts)
        q = torch.empty(d.shape, device=DEV, dtype=torch.float64)
        for k in range(self.D):
            for l in set(self.lev[ts][:, k]):
                m = torch.tensor(np.nonzero(self.lev[ts][:, k] == l)[0], device=DEV)
                q[m, :, k] = self.rules[self.mode_id[k], int(l)]["q"][d[m, :, k]]
        return q

    def slots(self, ts):
        o = torch.tensor(self.off[ts], device=DEV)
        return o[:, None] + torch.arange(int(self.nt[ts[0]]), device=DEV)[None, :]

    def on_grid(self, f):
        """f(q) at every grid point, in the order of the operator grids"""
        v = torch.empty(int(self.off[-1]), device=DEV, dtype=torch.float64)
        for _, ts in self.chunks(2e6):
            q = self.points(ts)
            v[self.slots(ts)] = f(q.reshape(-1, self.D)).reshape(q.shape[:2])
        return v

    def mul(self, key, which, x, only=None):
        """x (T, nv, N) times the matrices `which` of all modes of the key (or of one)"""
        T, nv, N = x.shape
        A = 1
        for j, k in enumerate(key):
            M = self.rules[k][which]
            if only is None or only == j:
                x = torch.matmul(M, x.reshape(-1, M.shape[1], A)).reshape(T, nv, N)
            A *= M.shape[0]
        return x

    def active(self, key, t):
        """modes of the key's entries in term t"""
        act = [k for k in range(self.D) if self.lev[t, k] or self.n[0] > 1]
        return act

    def scale(self, ts, key):
        """weight of a term times the 1 x 1 transforms of its one-point modes"""
        f = 1.0
        if self.n[0] == 1 and len(key) < self.D:
            r = self.rules[self.mode_id[0], 0]
            f = float(r["B"][0, 0] * r["Bt"][0, 0]) ** (self.D - len(key))
        return torch.tensor(self.wgt[ts], device=DEV) * f

    def hpsi(self, psi, local, budget=4e7):
        """sum_t W_t P_t^T B^T W local(...) B P_t psi, psi (nv, nb)"""
        nv = psi.shape[0]
        out = torch.zeros(self.nb, nv, device=DEV, dtype=torch.float64)
        for key, ts in self.chunks(budget / nv):
            r = self.rows(ts)
            x = psi[:, r].permute(1, 0, 2).contiguous()          # (T, nv, N)
            g = self.mul(key, "B", x)
            y = self.mul(key, "Bt", local(self, key, ts, g))
            y = y * self.scale(ts, key)[:, None, None]
            out.index_add_(0, r.reshape(-1), y.permute(0, 2, 1).reshape(-1, nv))
        return out.T.contiguous()


def _type1_local(V, ck):
    def local(S, key, ts, g):
        y = V(S.points(ts).reshape(-1, S.D)).reshape(len(ts), 1, -1) * g
        if ck is not None:
            full = S.n[0] > 1 or len(key) == S.D
            for j in range(len(key)):
                y = y + ck * S.mul(key, "D2", g, j)
            if not full:
                y = y + ck * (S.D - len(key)) * float(S.rules[S.mode_id[0], 0]["D2"][0, 0]) * g
        return y
    return local


def _model(pot, D, seed):
    if pot == "pes":
        return _pes(D, seed)
    lam = _lam(seed)

    def V(q):
        s = q * q
        v = 0.5 * s.sum(1)
        if q.shape[1] > 1:
            v = v + lam * (s[:, :-1] * q[:, 1:] - q[:, 1:] ** 3 / 3.0).sum(1)
        return v
    return V


def exact(case, seed):
    c = case
    if c["kind"] == "subspace":
        s = prepare(case, seed)
        return s["V"][:c["m"]] @ s["H"].T, s["U"] @ s["V"]
    if c["kind"] == "hpsi":
        S = _Sparse(c["D"], c["L"])
        return S.hpsi(_block(c["nvec"], S.nb, seed), _type1_local(_model(c["pot"], c["D"], seed), -0.5))
    if c["kind"] == "grad":
        S = _Sparse(c["D"], c["L"])
        psi, out = _block(c["nvec"], S.nb, seed), torch.empty(int(S.off[-1]), c["nvec"], device=DEV, dtype=torch.float64)
        w0 = float(S.rules[S.mode_id[0], 0]["wq"][0] * S.rules[S.mode_id[0], 0]["B"][0, 0] ** 2)
        for key, ts in S.chunks(4e7 / c["nvec"]):
            g = S.mul(key, "B", psi[:, S.rows(ts)].permute(1, 0, 2).contiguous())
            w = torch.ones(1, device=DEV, dtype=torch.float64)
            for k in key:
                w = (S.rules[k]["wq"][:, None] * w[None, :]).reshape(-1)
            w = w[None, :] * (torch.tensor(S.wgt[ts], device=DEV) * w0 ** (S.D - len(key)))[:, None]
            out[S.slots(ts)] = (w[:, None, :] * g * g).permute(0, 2, 1)
        return out
    if c["kind"] == "type1":
        S = _Sparse(c["D"], c["L"])
        der, fun = _type1_terms(c["D"], seed)

        def local(S, key, ts, g):
            # every mode takes part: one-point modes with their 1 x 1 derivative matrices
            q, y = S.points(ts).reshape(-1, S.D), torch.zeros_like(g)
            one = S.rules[S.mode_id[0], 0]
            lev = torch.tensor(S.lev[ts], device=DEV)
            pos = torch.cumsum((lev > 0).long(), 1) - 1

            def d(mode, which, x):
                z = x * float(one[which][0, 0])
                for j in range(len(key)):
                    m = torch.nonzero((lev[:, mode] > 0) & (pos[:, mode] == j)).reshape(-1)
                    if len(m):
                        z[m] = S.mul(key, which, x[m], j)
                return z
            for (i, j), f in zip(der, fun):
                u = g
                if i >= 0:
                    u = d(i, "D1", g) if j < 0 else d(i, "D2", g) if i == j else d(i, "D1", d(j, "D1", g))
                y = y + f(q).reshape(len(ts), 1, -1) * u
            return y
        return S.hpsi(_block(c["nvec"], S.nb, seed), local)
    if c["kind"] == "jacobi":
        A, Dm, a, Re, re = potentials.AMU, 0.2, 1.0, 3.0, 2.0
        s = math.sqrt(A * a * math.sqrt(2 * Dm / A))
        S = _Sparse(3, c["L"], [("ho", Re, s), ("ho", re, s), ("legendre", 0.0, 1.0)], nA=2)
        cp = 0.005 + 0.01 * np.random.default_rng(seed).random()

        def local(S, key, ts, g):
            q = S.points(ts)
            R, r, th = (q[:, None, :, k] for k in range(3))
            V = Dm * (1 - torch.exp(-a * (R - Re))) ** 2 + Dm * (1 - torch.exp(-a * (r - re))) ** 2 + cp * torch.cos(th) ** 2
            G = [1.0 / A, 1.0 / A, 1.0 / (A * R * R) + 1.0 / (A * r * r)]
            J = torch.sin(th)
            kin = 0.0
            for i in range(3):
                kin = kin + S.mul(key, "D1", J * G[i] * S.mul(key, "D1", g, i), i)
            return -0.5 * kin / J + V * g
        return S.hpsi(_block(c["nvec"], S.nb, seed), local)
    return _exact_field(c, seed)


def _exact_field(c, seed):
    """Dense matrices of every instance; None where they would be too large."""
    insts = _instances(c)
    rows = [int(_rows(d, l)) for d, l in insts]
    if max(rows) > 3000:
        return None
    from scipy.special import jv
    row0 = np.concatenate([[0], np.cumsum(rows)])
    psi, target = _states(row0, seed)
    eps, lo, hi = _field(c, seed), *_range(insts)
    E0, Esc = 0.5 * (hi + lo), 0.5 * (hi - lo)
    coef = jv(np.arange(200), Esc * DT)
    coef[1:] *= 2
    nmax = int(np.nonzero(np.abs(coef) > 1e-15)[0].max()) + 2
    ph = complex(math.cos(E0 * DT), -math.sin(E0 * DT))
    final, J, grad = [], 0.0, np.zeros(len(eps))
    for (d, l), r0, r1 in zip(insts, row0[:-1], row0[1:]):
        S = _Sparse(d, l)
        I = torch.eye(r1 - r0, device=DEV, dtype=torch.float64)
        H0 = S.hpsi(I, _type1_local(_model("hh", d, seed), -0.5)).T
        Mu = S.hpsi(I, _type1_local(lambda q: q.sum(1), None)).T.to(torch.complex128)
        H0 = H0.to(torch.complex128)

        def step(x, dx, e, sgn):
            """the Chebyshev step of H0 + e Mu and its derivative along e"""
            hs = lambda v: (H0 @ v + e * (Mu @ v) - E0 * v) / Esc
            w, t = [x, sgn * 1j * hs(x)], [dx, sgn * 1j * (hs(dx) + Mu @ x / Esc)]
            a, b = coef[0] * w[0] + coef[1] * w[1], coef[0] * t[0] + coef[1] * t[1]
            for k in range(2, nmax):
                w, t = ([w[1], w[0] + 2j * sgn * hs(w[1])],
                        [t[1], t[0] + 2j * sgn * (hs(t[1]) + Mu @ w[1] / Esc)])
                a, b = a + coef[k] * w[1], b + coef[k] * t[1]
            p = ph if sgn < 0 else ph.conjugate()
            return a * p, b * p
        at = [psi[0, r0:r1]]
        for e in eps:
            x = at[-1]
            for _ in range(c["steps"]):
                x, _ = step(x, torch.zeros_like(x), e, -1)
            at.append(x)
        final.append(at[-1])
        if c["kind"] == "fieldgrad":
            ov = torch.sum(target[0, r0:r1].conj() * at[-1])
            J += abs(ov.item()) ** 2
            lam = ov * target[0, r0:r1]
            for s in range(len(eps) - 1, -1, -1):
                x, dx = at[s], torch.zeros_like(at[s])
                for _ in range(c["steps"]):
                    x, dx = step(x, dx, eps[s], -1)
                grad[s] += 2.0 * torch.sum(lam.conj() * dx).item().real
                for _ in range(c["steps"]):
                    lam, _ = step(lam, torch.zeros_like(lam), eps[s], 1)
    if c["kind"] == "field":
        return torch.cat(final)[None, :]
    return dict(J=J, grad=grad)
