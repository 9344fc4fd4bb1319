"""Request loop for Fock builds on one GPU, with continuous batching.

A request is one molecule (basis in the liberi_setup convention) and the
densities of its SCF-like iterations.  The loop admits requests as they
arrive, while a slot and enough HBM are free (the admission test uses an
estimate of the handle's device footprint: shell pairs, primitive pairs,
quartet tables, D and F).  An admitted request gets its own handle -- its
shell pairs stay resident in HBM for all its iterations -- and its own HIP
stream, on which every iteration is enqueued at once: density upload, Fock
build, Fock download.  Requests admitted together therefore run concurrently
on the device; a request that arrives while others run is admitted as soon
as one of them retires.  Latency is measured from arrival to the moment the
last iteration's Fock matrix is in host memory.

The Schwarz integrals of each molecule are computed on the GPU at admission
(liberi_c_schwarz), so a request needs nothing from the host but its basis
and densities.
"""
from __future__ import annotations

import collections
import math
import time
from dataclasses import dataclass, field

import numpy as np

from . import hipmem, liberi
from .caseio import Basis


@dataclass
class Request:
    rid: int
    arrival: float  # seconds after the start of the stream
    basis: Basis
    densities: list  # packed densities, one per iteration
    tau: float = 0.0  # mixed-precision switch (0 = FP64)


@dataclass
class Result:
    rid: int
    arrival: float
    admitted: float
    done: float
    nbf: int
    quartets: int
    device_bytes: int
    iterations: int
    focks: list = field(default_factory=list)

    @property
    def latency(self) -> float:
        return self.done - self.arrival


def _quartet_bounds(basis: Basis) -> tuple[int, int]:
    """Upper bounds of the quartets that survive screening, all of them and those
    with a (pd| or (dd| pair: every quartet of a small basis, else those whose
    pairs' Gaussian decay exp(-ab/(a+b) R^2), at the smallest exponents, leaves
    more than exp(-40) = 4e-18 of 5e-11 (a margin of 1e7 for what stands before
    the exponentials)."""
    nsh = basis.nsh
    npairs = nsh * (nsh + 1) // 2
    loc, k = np.asarray(basis.sh_loc, dtype=np.int64) - 1, np.asarray(basis.contr_num, dtype=np.int64)
    expo, xyz = np.asarray(basis.exponents), np.asarray(basis.coords).reshape(-1, 3)
    atom = np.asarray(basis.atom_num) - 1
    every_quartet = npairs * (npairs + 1) // 2
    # (a basis out of its arrays is the setup's to refuse)
    if npairs <= 4096 or np.any((k < 1) | (loc < 0) | (loc + k > expo.size) | (atom < 0) | (atom >= len(xyz))):
        return every_quartet, every_quartet
    e = np.array([np.min(expo[i:i + n]) for i, n in zip(loc, k)])
    if not (np.all(np.isfinite(e) & (e > 0)) and np.all(np.isfinite(xyz))):
        return every_quartet, every_quartet
    # ordered pairs by decay, in steps of 0.1 rounded down, some rows at a time
    L = np.asarray(basis.ang_mom) - 1
    centre = xyz[atom]
    sq = np.sum(centre * centre, axis=1)
    every, pd = np.zeros(402), np.zeros(402)
    for i in range(0, nsh, 512):
        r = slice(i, i + 512)
        r2 = np.maximum(sq[r, None] + sq - 2.0 * centre[r] @ centre.T, 0.0)
        step = np.minimum(10.0 * e[r, None] * e / (e[r, None] + e) * r2, 401.0).astype(np.int64)
        hi, lo = np.maximum(L[r, None], L), np.minimum(L[r, None], L)
        every += np.bincount(step.ravel(), minlength=402)
        pd += np.bincount(step[(hi == 2) & (lo >= 1)], minlength=402)
    partners = np.cumsum(every[:401])[::-1]
    return int(every[:401] @ partners / 8) + npairs * nsh, int(pd[:401] @ partners / 4) + npairs * nsh


def estimate_device_bytes(basis: Basis) -> int:
    """Upper estimate of the HBM a handle holds for this basis (bytes)."""
    L = np.asarray(basis.ang_mom) - 1
    k = np.asarray(basis.contr_num, dtype=np.int64)
    nsh = basis.nsh
    npairs = nsh * (nsh + 1) // 2
    nprim = int((np.sum(k) ** 2 + np.sum(k * k)) // 2)
    ntri = basis.num_bas * (basis.num_bas + 1) // 2
    per_l = np.bincount(L, minlength=4).astype(np.int64)
    # pairs of each pair class (la >= lb)
    pcount = {(a, b): (per_l[a] * (per_l[a] + 1) // 2 if a == b else per_l[a] * per_l[b])
              for a in range(4) for b in range(a + 1)}
    # each class keeps, per kept row, a few segments (16 B) and a tile (24 B) in
    # each of up to five tables; a pair class serves as the rows of at most 10
    # classes.  Long rows have a tile every 512, 1024, 4096 and 16384 quartets
    # (more where lanes share quartets, in classes of few), and classes of few
    # quartets 2048 of one workgroup step at most; the work items of the fused
    # launch (24 B) hold at least 32 quartets.
    quartets, fused = _quartet_bounds(basis)
    tables = (10 * (6 * 16 + 5 * 24) * npairs + 24 * min(quartets // 64, 55 * 2048)
              + 24 * quartets * (1 / 512 + 1 / 1024 + 1 / 4096 + 1 / 16384) + 24 * fused / 32)
    # the density and the Coulomb sums by shell pair (twice each), the square
    # density and exchange sums
    ncart = [1, 3, 6, 10]
    by_pair = sum(n * ncart[a] * ncart[b] for (a, b), n in pcount.items())
    return int(64 * (npairs + nprim) + 8 * (3 * ntri + 4 * by_pair + 2 * basis.num_bas ** 2) + tables + 4 * basis.num_bas
               + (1 << 20))


def percentile(x, q: float) -> float:
    """Nearest-rank percentile (q in 0..100)."""
    s = sorted(x)
    if not s:
        return float("nan")
    r = max(1, math.ceil(q / 100.0 * len(s)))
    return float(s[r - 1])


class _Slot:
    def __init__(self, req: Request, t_admit: float, need: int):
        self.req = req
        self.t_admit = t_admit
        self.need = need
        b = req.basis
        sw = liberi.schwarz(b)
        self.h = liberi.Handle()
        self.h.setup(b.with_schwarz(sw))
        if req.tau > 0:
            self.h.set_option(liberi.OPT_FP32_TAU, req.tau)
        self.n = b.ntri
        self.stream = hipmem.Stream()
        # one allocation on each side: densities and Fock matrices of every
        # iteration in pinned memory, one of each on the device
        self.device = hipmem.DeviceArray(2 * self.n)
        self.D, self.F = self.device.part(0, self.n), self.device.part(self.n, self.n)
        k = len(req.densities)
        self.host = hipmem.PinnedArray(2 * k * self.n)
        self.hD = [self.host.part(i * self.n, self.n) for i in range(k)]
        self.hF = [self.host.part((k + i) * self.n, self.n) for i in range(k)]
        for p, d in zip(self.hD, req.densities):
            p.array[:] = d
        st = self.h.stats()
        self.quartets = int(st["total_quartets"])
        self.device_bytes = int(st["device_bytes"])
        # every iteration on the request's stream: D in, build, F out
        for pd, pf in zip(self.hD, self.hF):
            self.D.copy_from_async(pd, self.stream)
            self.h.fock_build_device(self.D.address, self.F.address, self.n, self.stream.address)
            self.F.copy_to_async(pf, self.stream)
        self.event = hipmem.Event()
        self.event.record(self.stream)

    def finish(self, keep: bool) -> list:
        focks = [pf.array.copy() for pf in self.hF] if keep else []
        self.device_bytes = max(self.device_bytes, int(self.h.stats()["device_bytes"]))
        self.h.destroy()
        self.event.destroy()
        self.stream.destroy()
        self.device.free()
        for p in self.hD + self.hF:
            p.free()
        self.host.free()
        return focks


class Server:
    """Continuous-batching request loop on the current GPU.

    max_active -- requests on the device at once (slots);
    hbm_budget -- bytes of HBM the admitted requests may hold together
                  (default: half of the free HBM when the server starts).
    """

    def __init__(self, max_active: int = 4, hbm_budget: int | None = None, keep_focks: bool = True):
        self.max_active = max_active
        if hbm_budget is None:
            free, _ = hipmem.device_memory()
            hbm_budget = free // 2
        self.hbm_budget = hbm_budget
        self.keep_focks = keep_focks
        self.peak_active = 0  # most requests on the device at once in the last run
        self.peak_bytes = 0   # most estimated HBM held at once in the last run

    def run(self, requests: list) -> list:
        pending = collections.deque(sorted(requests, key=lambda r: r.arrival))
        queue = collections.deque()
        active = []
        used = 0
        results = []
        self.peak_active = self.peak_bytes = 0
        t0 = time.perf_counter()
        while pending or queue or active:
            now = time.perf_counter() - t0
            while pending and pending[0].arrival <= now:
                req = pending.popleft()
                queue.append((req, estimate_device_bytes(req.basis)))
            progressed = False
            # retire finished requests first: their memory and slots go to the queue
            for s in list(active):
                if s.event.done():
                    t_done = time.perf_counter() - t0
                    focks = s.finish(self.keep_focks)
                    results.append(Result(s.req.rid, s.req.arrival, s.t_admit, t_done, s.req.basis.num_bas,
                                          s.quartets, s.device_bytes, len(s.req.densities), focks))
                    active.remove(s)
                    used -= s.need
                    progressed = True
            # admit while a slot and the memory allow (a lone request is always admitted)
            while queue and len(active) < self.max_active:
                req, need = queue[0]
                if active and used + need > self.hbm_budget:
                    break
                queue.popleft()
                active.append(_Slot(req, time.perf_counter() - t0, need))
                used += need
                self.peak_active = max(self.peak_active, len(active))
                self.peak_bytes = max(self.peak_bytes, used)
                progressed = True
            if not progressed:
                wait = 0.0005
                if not active and not queue and pending:
                    wait = max(0.0, pending[0].arrival - (time.perf_counter() - t0))
                time.sleep(min(wait, 0.05))
        results.sort(key=lambda r: r.rid)
        return results


def summarize(results: list, wall: float | None = None) -> dict:
    lat = [r.latency for r in results]
    builds = sum(r.iterations for r in results)
    t_first = min(r.arrival for r in results)
    t_last = max(r.done for r in results)
    span = wall if wall is not None else (t_last - t_first)
    return {"requests": len(results), "p50_latency_s": percentile(lat, 50), "p99_latency_s": percentile(lat, 99),
            "mean_latency_s": float(np.mean(lat)), "span_s": span, "builds": builds,
            "builds_per_s": builds / span, "quartets_per_s": sum(r.quartets * r.iterations for r in results) / span}


def scf_like_densities(nbf: int, nocc: int, iterations: int, seed: int, eps0: float = 0.05) -> list:
    """Densities of SCF-like iterations: D_k = 2 Q_k Q_k^T (packed), Q_k the
    orthonormalised C + eps_k G_k with C a seeded orthonormal n x nocc block and
    eps_k = eps0 / (k + 1) (the perturbation shrinks as an SCF converges)."""
    rng = np.random.default_rng(seed)
    c, _ = np.linalg.qr(rng.standard_normal((nbf, nocc)))
    il = np.tril_indices(nbf)
    out = []
    for k in range(iterations):
        q, _ = np.linalg.qr(c + eps0 / (k + 1) * rng.standard_normal(c.shape))
        out.append(np.ascontiguousarray((2.0 * q @ q.T)[il]))
    return out


def request_stream(n: int, rate: float, seed: int, iterations: int = 10, tau: float = 0.0,
                   atoms: tuple = (10, 200)) -> list:
    """Poisson arrivals (rate per second) of random H/C/N/O clusters of
    U{atoms} atoms (gms_liberi_amd.configs.cluster), each with its SCF-like
    densities (N_electrons/2 occupied)."""
    from .configs import cluster

    rng = np.random.default_rng(seed)
    t = 0.0
    reqs = []
    for i in range(n):
        t += rng.exponential(1.0 / rate) if i else 0.0
        natoms = int(rng.integers(atoms[0], atoms[1] + 1))
        case = cluster(natoms, seed * 1000 + i)
        nocc = int(round(float(np.sum(case.density[[j * (j + 3) // 2 for j in range(case.basis.num_bas)]])) / 2))
        dens = scf_like_densities(case.basis.num_bas, nocc, iterations, seed * 1000 + i)
        reqs.append(Request(i, t, case.basis, dens, tau))
    return reqs
