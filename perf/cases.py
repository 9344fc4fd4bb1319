"""Workloads of the Fock build that its users run, through the public entry points.

A case names an entry point (``call``), a molecule family of
``gms_liberi_amd.configs`` (``mol``, ``natoms``, ``basis_seed``) and the options
of the call.  The seed of ``prepare`` moves every atom by about 0.01 bohr (one
step of a geometry optimisation) and draws the density.

  device   one SCF iteration with D and F resident in HBM
  host     one SCF iteration on host arrays, the reference's protocol
  uhf      the two Fock matrices of an unrestricted iteration, host arrays
  share    this rank's partial F of a build split over ``ranks`` processes
  schwarz  the Schwarz integrals of a new geometry
  serve    a batch of requests through the serving loop: Schwarz integrals,
           setup and the SCF-like iterations of every molecule
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gms_liberi_amd import configs, liberi, serving
from gms_liberi_amd.census import CLASS_L


def _case(call, mol, natoms, basis_seed, **more):
    return {"call": call, "mol": mol, "natoms": natoms, "basis_seed": basis_seed, "ranks": 1, "rank": 0, "tau": 0.0,
            "iterations": 1, "requests": 0, **more}


def listed():
    return [
        # the smallest molecule (13 functions, s and p): launches and the longest primitive chain
        {"name": "water", **_case("device", "water", 3, 11)},
        # a small molecule through the reference's own host-array protocol (42 functions, s, p, d)
        {"name": "ethane_host", **_case("host", "ethane", 8, 12)},
        # a small odd-sized molecule with every f class, most of them with few quartets (93 functions)
        {"name": "chain3_host", **_case("host", "cn_chain", 3, 14)},
        # an ordinary small molecule: 12 heavy atoms, 180 functions
        {"name": "cage12", **_case("device", "cage", 12, 13)},
        # the mixed FP32/FP64 form at the switch the serving stream uses, odd size (345 functions)
        {"name": "cage23_mixed", **_case("device", "cage", 23, 13, tau=1e-6)},
        # an unrestricted iteration of a 17-atom H/C/N/O cluster
        {"name": "cluster17_uhf", **_case("uhf", "cluster", 17, 5)},
        # an odd-sized H/C/N/O cluster of the request stream's recipe
        {"name": "cluster41", **_case("device", "cluster", 41, 7)},
        # f functions in earnest: the 20-atom C/N chain (620 functions)
        {"name": "chain20", **_case("device", "cn_chain", 20, 14)},
        # the largest: the 60-carbon cage (900 functions, 262M quartets)
        {"name": "c60", **_case("device", "c60", 60, 13)},
        # one process's share of that build when eight split it
        {"name": "c60_share", **_case("share", "c60", 60, 13, ranks=8, rank=5)},
        # Schwarz integrals of a new geometry, f functions among them
        {"name": "schwarz_chain20", **_case("schwarz", "cn_chain", 20, 14)},
        # new molecules arriving together: all of setup is paid per request
        {"name": "serve3", **_case("serve", "cluster", 12, 21, requests=3, iterations=4)},
    ]


def draw(rng):
    seed = rng.randrange(1 << 20)

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    call = rng.choice(["device", "device", "device", "host", "host", "uhf", "share", "schwarz", "serve"])
    if call == "uhf":
        mol = rng.choice(["ethane", "cluster", "cage"])
        return _case(call, mol, 8 if mol == "ethane" else size(4, 30), seed)
    if call == "serve":
        return _case(call, "cluster", size(6, 24), seed, requests=rng.randrange(1, 5), iterations=rng.randrange(2, 6))
    if call == "share":
        ranks = rng.choice([2, 3, 4, 8])
        mol = rng.choice(["cage", "cn_chain", "cluster"])
        return _case(call, mol, size(12, 58) if mol != "cn_chain" else size(6, 20), seed, ranks=ranks,
                     rank=rng.randrange(ranks))
    mol = rng.choice(["water", "ethane", "cage", "cage", "cluster", "cluster", "cn_chain", "cn_chain"])
    natoms = {"water": 3, "ethane": 8, "cage": size(4, 58), "cluster": size(3, 60), "cn_chain": size(3, 20)}[mol]
    tau = 1e-6 if call == "device" and rng.random() < 0.15 else 0.0
    return _case(call, mol, natoms, seed, tau=tau)


# ------------------------------------------------------------------ inputs
def _molecule(mol, natoms, basis_seed):
    if mol == "water":
        return configs.water(basis_seed)
    if mol == "ethane":
        return configs.ethane(basis_seed)
    if mol == "c60":
        return configs.c60(basis_seed)
    if mol == "cage":
        return configs.c60_fragment(natoms, basis_seed)
    if mol == "cn_chain":
        return configs.cn_chain(basis_seed, natoms)
    return configs.cluster(natoms, basis_seed)


def _occupied(case):
    """Occupied orbitals of the generator's density (its trace is twice that)."""
    b = case.basis
    return int(round(sum(case.density[j * (j + 3) // 2] for j in range(b.num_bas)) / 2))


def _inputs(case, seed):
    """[(basis, packed densities)] of the case: one molecule, or one per request."""
    rng = np.random.default_rng([seed, 77])
    got = []
    for k in range(max(1, case["requests"])):
        natoms = case["natoms"] + 3 * k
        c = _molecule(case["mol"], natoms, case["basis_seed"] + k)
        b = c.basis
        b.coords[:] = b.coords + 0.01 * rng.standard_normal(b.coords.shape)
        nocc = min(_occupied(c), b.num_bas)
        if case["call"] == "serve":
            dens = serving.scf_like_densities(b.num_bas, nocc, case["iterations"], int(rng.integers(1 << 30)))
        elif case["call"] == "schwarz":
            dens = []
        else:
            dens = [configs.random_density(b.num_bas, nocc, rng)]
            if case["call"] == "uhf":  # spin densities of nocc and nocc - 1 electrons
                dens = [0.5 * dens[0], 0.5 * configs.random_density(b.num_bas, max(1, nocc - 1), rng)]
        got.append((b, dens))
    return got


_stream = None


def _program_stream():
    """The one compute stream of the program."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def prepare(case, seed):
    given = _inputs(case, seed)
    b, dens = given[0]
    state = {"call": case["call"], "basis": b}
    if case["call"] == "schwarz":
        return state
    if case["call"] == "serve":
        state["requests"] = [serving.Request(i, 0.0, x, d) for i, (x, d) in enumerate(given)]
        return state
    h = liberi.Handle()
    h.setup(b.with_schwarz(liberi.schwarz(b)), case["rank"], case["ranks"])
    if case["tau"] > 0.0:
        h.set_option(liberi.OPT_FP32_TAU, case["tau"])
    state["handle"] = h
    if case["call"] in ("host", "uhf"):
        state["density"] = dens
        state["fock"] = np.empty(b.ntri)
        return state
    state["D"] = torch.from_numpy(dens[0]).cuda()
    state["F"] = torch.empty_like(state["D"])
    state["stream"] = _program_stream()
    return state


def run(state):
    call = state["call"]
    if call == "schwarz":
        return liberi.schwarz(state["basis"])
    if call == "serve":
        return [r.focks for r in serving.Server(max_active=4).run(state["requests"])]
    h = state["handle"]
    if call == "uhf":
        return list(h.fock_build_uhf(*state["density"]))
    if call == "host":
        return h.fock_build(state["density"][0], state["fock"])
    d, f = state["D"], state["F"]
    h.fock_build_device(d.data_ptr(), f.data_ptr(), d.numel(), state["stream"].cuda_stream)
    return f


# -------------------------------------------------------------------- work
def _ncart(l):
    return (l + 1) * (l + 2) // 2


def _nrange(l0, l1):
    return sum(_ncart(l) for l in range(l0, l1 + 1))


def _table_flops(ni, nk):
    return 3 * (ni - 1) + 5 * ni * (nk - 1)


def _class_flops(c, quartets, prims, spins):
    """Rys quadrature of (e0|f0) per primitive quartet (FMA = 2; two degree-7
    polynomials per root), the horizontal recurrence and the six digestion
    blocks (two Coulomb, four exchange per spin) per contracted quartet."""
    la, lb, lc, ld = CLASS_L[c]
    nr = (la + lb + lc + ld) // 2 + 1
    ne, nf = _nrange(la, la + lb), _nrange(lc, lc + ld)
    per_prim = 15 + nr * (28 + 22 + 3 * _table_flops(la + lb + 1, lc + ld + 1) + 3 * ne * nf)
    nab, ncd = _ncart(la) * _ncart(lb), _ncart(lc) * _ncart(ld)
    hrr = sum(2 * _nrange(la, la + lb - j) * _ncart(j) * nf for j in range(1, lb + 1))
    hrr += sum(2 * nab * _nrange(lc, lc + ld - j) * _ncart(j) for j in range(1, ld + 1))
    return prims * per_prim + quartets * (hrr + (4 + 8 * spins) * nab * ncd)


def work(case):
    nbytes = flops = 0.0
    spins = 2 if case["call"] == "uhf" else 1
    for b, dens in _inputs(case, 0):
        l, k = b.ang_mom.astype(np.int64) - 1, b.contr_num.astype(np.int64)
        if case["call"] == "schwarz":
            nbytes += 24 * int(k.sum()) + 8 * b.schwrz.size
            for la in range(4):
                for lb in range(la + 1):
                    ka, kb = k[l == la] ** 2, k[l == lb] ** 2
                    # sum over pairs of nprim^2, A >= B within one angular momentum
                    n = ((ka.sum() ** 2 + (ka ** 2).sum()) / 2) if la == lb else ka.sum() * kb.sum()
                    per = 15 + (la + lb + 1) * (50 + 3 * _table_flops(la + lb + 1, la + lb + 1)
                                                + 3 * _ncart(la) * _ncart(lb))
                    flops += float(n) * per
            continue
        h = liberi.Handle()
        h.setup(b.with_schwarz(liberi.schwarz(b)), case["rank"], case["ranks"])
        st = h.stats()
        h.destroy()
        builds = max(1, len(dens)) if case["call"] == "serve" else 1
        npairs = b.nsh * (b.nsh + 1) // 2
        nbytes += builds * (16.0 * spins * b.ntri + 64.0 * (npairs + st["prim_pairs"]))
        for c in range(len(CLASS_L)):
            flops += builds * float(_class_flops(c, int(st["quartets"][c]), int(st["prim_quartets"][c]), spins))
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------- exact
# The same integrals by quadrature over t in (ab|cd) ~ int_0^1 exp(-X t^2)
# Ix Iy Iz dt with 64 Gauss-Legendre points on [0, min(1, sqrt(50 / X))], all
# primitive quartets, no screening.
_ORDER = {0: ["", ], 1: ["x", "y", "z"], 2: ["xx", "yy", "zz", "xy", "xz", "yz"],
          3: ["xxx", "yyy", "zzz", "xxy", "xxz", "xyy", "yyz", "xzz", "yzz", "xyz"]}


def _components(l):
    return [tuple(s.count(a) for a in "xyz") for s in _ORDER[l]]


def _scale(c):
    """Normalisation of a mixed component relative to x^l: sqrt of the ratio of double factorials."""
    def df(n):
        return math.prod(range(2 * n - 1, 0, -2)) if n > 0 else 1
    return math.sqrt(df(sum(c)) / (df(c[0]) * df(c[1]) * df(c[2])))


class _Pairs:
    """Shell pairs of one (la, lb), flattened over primitive pairs, on the device."""

    def __init__(self, b, la, lb, dev):
        l = b.ang_mom - 1
        coef = (b.coef_s, b.coef_p, b.coef_d, b.coef_f)
        xyz = b.coords.reshape(-1, 3)
        self.shells, rows = [], []
        for i in np.flatnonzero(l == la):
            for j in np.flatnonzero(l == lb):
                if la == lb and j > i:
                    continue
                self.shells.append((int(i), int(j)))
                a0, b0 = b.sh_loc[i] - 1, b.sh_loc[j] - 1
                ra, rb = xyz[b.atom_num[i] - 1], xyz[b.atom_num[j] - 1]
                for u in range(b.contr_num[i]):
                    for v in range(b.contr_num[j]):
                        x, y = b.exponents[a0 + u], b.exponents[b0 + v]
                        p = x + y
                        c = coef[la][a0 + u] * coef[lb][b0 + v] * math.exp(-x * y / p * float((ra - rb) @ (ra - rb)))
                        rows.append([len(self.shells) - 1, p, c / p, *((x * ra + y * rb) / p), *ra, *(ra - rb)])
        self.la, self.lb, self.n = la, lb, len(self.shells)
        r = np.array(rows).reshape(-1, 12)
        self.row = torch.tensor(r, dtype=torch.float64, device=dev)
        self.idx = torch.tensor(r[:, 0].astype(np.int64), device=dev)
        self.comps = [(ca, cb) for ca in _components(la) for cb in _components(lb)]
        self.scales = torch.tensor([_scale(ca) * _scale(cb) for ca, cb in self.comps], dtype=torch.float64, device=dev)


def _tables(P, Q, la, lb, lc, ld, dim, t2, hp, hq, ipq, p, q, g00):
    """I[a][b][c][d] of one direction: vertical recurrence, then both transfers."""
    pq = P[..., 3 + dim] - Q[..., 3 + dim]
    fa, fc = q * ipq * t2, p * ipq * t2
    c0, c1 = (P[..., 3 + dim] - P[..., 6 + dim]) - fa * pq, (Q[..., 3 + dim] - Q[..., 6 + dim]) + fc * pq
    b00, b10, b01 = 0.5 * t2 * ipq, hp * (1 - fa), hq * (1 - fc)
    ni, nk = la + lb + 1, lc + ld + 1
    g = [[None] * nk for _ in range(ni)]
    for i in range(ni):
        g[i][0] = g00 if i == 0 else c0 * g[i - 1][0] + ((i - 1) * b10 * g[i - 2][0] if i > 1 else 0.0)
    for k in range(1, nk):
        for i in range(ni):
            v = c1 * g[i][k - 1]
            if k > 1:
                v = v + (k - 1) * b01 * g[i][k - 2]
            if i > 0:
                v = v + i * b00 * g[i - 1][k - 1]
            g[i][k] = v
    ab, cd = P[..., 9 + dim], Q[..., 9 + dim]
    bra = [g]
    for j in range(lb):
        bra.append([[bra[j][i + 1][k] + ab * bra[j][i][k] for k in range(nk)] for i in range(ni - j - 1)])
    out = []
    for a in range(la + 1):
        for j in range(lb + 1):
            ket = [bra[j][a]]
            for m in range(ld):
                ket.append([ket[m][k + 1] + cd * ket[m][k] for k in range(nk - m - 1)])
            out.append(torch.stack([ket[m][c] for c in range(lc + 1) for m in range(ld + 1)]))
    return out


_NODES = np.polynomial.legendre.leggauss(64)


def _quartets(P, Q, bra, ket):
    """Primitive integrals [ab][cd, ...] for broadcastable primitive-pair rows P, Q (... , 12)."""
    dev = P.device
    x, w = (torch.tensor(v, dtype=torch.float64, device=dev) for v in (0.5 * (_NODES[0] + 1), 0.5 * _NODES[1]))
    P, Q = P.unsqueeze(-2), Q.unsqueeze(-2)  # nodes on the last axis
    p, q = P[..., 1], Q[..., 1]
    ipq = 1.0 / (p + q)
    X = p * q * ipq * ((P[..., 3:6] - Q[..., 3:6]) ** 2).sum(-1)
    end = torch.sqrt(50.0 / torch.clamp(X, min=50.0))
    t2 = (end * x) ** 2
    weight = 2 * math.pi ** 2.5 * P[..., 2] * Q[..., 2] * torch.sqrt(ipq) * end * w * torch.exp(-X * t2)
    la, lb, lc, ld = bra.la, bra.lb, ket.la, ket.lb
    one = torch.ones_like(weight)
    tab = [_tables(P, Q, la, lb, lc, ld, d, t2, 0.5 / p, 0.5 / q, ipq, p, q, weight if d == 2 else one)
           for d in range(3)]
    at = [torch.tensor([c[d] * (ld + 1) + e[d] for c, e in ket.comps], device=dev) for d in range(3)]
    for ca, cb in bra.comps:
        v = None
        for d in range(3):
            f = tab[d][ca[d] * (lb + 1) + cb[d]][at[d]]
            v = f if v is None else v * f
        yield v.sum(-1)


def _eri(b, dev):
    """Every integral (ij|kl) of the basis."""
    n = b.num_bas
    first = b.atom_loc - 1
    eri = torch.zeros(n, n, n, n, dtype=torch.float64, device=dev)
    ls = sorted(set((b.ang_mom - 1).tolist()))
    pairs = [_Pairs(b, la, lb, dev) for la in ls for lb in ls if lb <= la]
    for x, bra in enumerate(pairs):
        for ket in pairs[:x + 1]:
            per = 64 * 8 * (len(ket.comps) * 4 + 4 * (bra.la + 1) * (bra.lb + 1) * (ket.la + 1) * (ket.lb + 1))
            step = max(1, int(4e9 / (per * len(ket.row))))
            val = torch.zeros(len(bra.comps), bra.n, len(ket.comps), ket.n, dtype=torch.float64, device=dev)
            for s in range(0, len(bra.row), step):
                P = bra.row[s:s + step, None, :]
                for i, v in enumerate(_quartets(P, ket.row[None], bra, ket)):  # (cd, prim ab, prim cd)
                    c = torch.zeros(len(ket.comps), v.shape[1], ket.n, dtype=torch.float64, device=dev)
                    c.index_add_(2, ket.idx, v)
                    val[i].index_add_(0, bra.idx[s:s + step], c.transpose(0, 1).contiguous())
            val *= bra.scales[:, None, None, None] * ket.scales[None, None, :, None]

            def funcs(t):
                na, nb = len(_components(t.la)), len(_components(t.lb))
                i = np.array([[first[A] + c // nb for A, _ in t.shells] for c in range(na * nb)])
                j = np.array([[first[B] + c % nb for _, B in t.shells] for c in range(na * nb)])
                return torch.tensor(i.reshape(-1), device=dev), torch.tensor(j.reshape(-1), device=dev)

            (i, j), (k, l) = funcs(bra), funcs(ket)
            flat = val.reshape(len(i), len(k))
            for u, v in ((i, j), (j, i)):
                for r, s in ((k, l), (l, k)):
                    eri[u[:, None], v[:, None], r[None], s[None]] = flat
                    eri[r[:, None], s[:, None], u[None], v[None]] = flat.t()
    return eri


def _full(packed, n, dev):
    m = torch.zeros(n, n, dtype=torch.float64, device=dev)
    i, j = torch.tril_indices(n, n, device=dev)
    m[i, j] = m[j, i] = torch.from_numpy(packed).to(dev)
    return m


def _fock(eri, d_coulomb, d_exchange, weight):
    n = d_coulomb.shape[0]
    jm = (eri.reshape(n * n, n * n) @ d_coulomb.reshape(-1)).reshape(n, n)
    km = (eri.permute(0, 2, 1, 3).reshape(n * n, n * n) @ d_exchange.reshape(-1)).reshape(n, n)
    f = jm - weight * km
    f = 2 * f - torch.diag(torch.diag(f))
    i, j = torch.tril_indices(n, n, device=f.device)
    return f[i, j].contiguous()


def exact(case, seed):
    given = _inputs(case, seed)
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if case["call"] == "schwarz":
        b = given[0][0]
        if b.natoms > 24:
            return None
        out = torch.zeros(b.nsh * (b.nsh + 1) // 2, dtype=torch.float64, device=dev)
        for la in range(4):
            for lb in range(la + 1):
                t = _Pairs(b, la, lb, dev)
                if not t.n:
                    continue
                # primitive quartets of (ab|ab), the pairs of one primitive count together
                count = torch.bincount(t.idx, minlength=t.n).cpu()
                start = torch.cumsum(count, 0) - count
                for n in sorted(set(count.tolist())):
                    which = torch.nonzero(count == n).flatten()
                    step = max(1, int(2e9 / (64 * 8 * n * n * (4 * len(t.comps) + 4 * (la + 1) ** 2 * (lb + 1) ** 2))))
                    for s in range(0, len(which), step):
                        pick = which[s:s + step]
                        P = t.row[(start[pick, None] + torch.arange(n)).to(dev)]
                        best = torch.zeros(len(pick), dtype=torch.float64, device=dev)
                        for k, v in enumerate(_quartets(P[:, :, None], P[:, None], t, t)):
                            best = torch.maximum(best, (v[k].sum((-1, -2)) * t.scales[k] ** 2).abs())
                        at = [max(t.shells[m]) * (max(t.shells[m]) + 1) // 2 + min(t.shells[m]) for m in pick.tolist()]
                        out[torch.tensor(at, device=dev)] = torch.sqrt(best)
        return out
    if case["ranks"] > 1 or max(b.num_bas for b, _ in given) > 100:
        return None
    got = []
    for b, dens in given:
        eri = _eri(b, dev)
        full = [_full(d, b.num_bas, dev) for d in dens]
        if case["call"] == "uhf":
            return [_fock(eri, full[0] + full[1], d, 1.0) for d in full]
        got.append([_fock(eri, d, d, 0.5) for d in full])
    return got if case["call"] == "serve" else got[0][0]
