"""Unrestricted Fock matrices (the reference's FOCK_B, registered in its MDI
plugin but never computed, src/interface/liberi_mdi_api.F90:404-409).

Pinned by the closed forms Fa = S o (J[Da+Db] - K[Da]),
Fb = S o (J[Da+Db] - K[Db]) with J and K from the oracle's full ERI tensor,
and by the RHF limit Da = Db = D/2.
"""
from pathlib import Path

import numpy as np
import pytest

from gms_liberi_amd import liberi
from gms_liberi_amd.caseio import Case
from tests.test_oracle import unpack

GOLD = Path(__file__).resolve().parent / "golden"
CUT = 5.00000000000000018e-11


def _spin_densities(n, rng, occ_a, occ_b):
    q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    il = np.tril_indices(n)
    da = (q[:, :occ_a] @ q[:, :occ_a].T)[il]
    db = (q[:, :occ_b] @ q[:, :occ_b].T)[il]
    return np.ascontiguousarray(da), np.ascontiguousarray(db)


@pytest.mark.gpu
def test_uhf_closed_form(oracle):
    case = Case.load_npz(GOLD / "cfg_water.npz")
    b = case.basis.with_schwarz(np.full(case.basis.nsh * (case.basis.nsh + 1) // 2, 1e10))  # no screening
    n = b.num_bas
    eri = np.zeros((n, n, n, n))
    loc = b.atom_loc - 1
    size = b.ang_mom * (b.ang_mom + 1) // 2
    for i in range(b.nsh):
        for j in range(b.nsh):
            for k in range(b.nsh):
                for l in range(b.nsh):
                    eri[loc[i]:loc[i] + size[i], loc[j]:loc[j] + size[j], loc[k]:loc[k] + size[k],
                        loc[l]:loc[l] + size[l]] = oracle.quartet(b, i, j, k, l)
    eri[np.abs(eri) < CUT] = 0.0
    da, db = _spin_densities(n, np.random.default_rng(8), 5, 4)
    Da, Db = unpack(da), unpack(db)
    J = np.einsum("ijkl,kl->ij", eri, Da + Db)
    S = 2.0 - np.eye(n)
    il = np.tril_indices(n)
    want_a = (S * (J - np.einsum("ikjl,kl->ij", eri, Da)))[il]
    want_b = (S * (J - np.einsum("ikjl,kl->ij", eri, Db)))[il]
    h = liberi.Handle()
    h.setup(b)
    fa, fb = h.fock_build_uhf(da, db)
    h.destroy()
    scale = max(1.0, float(np.max(np.abs(want_a))))
    assert np.max(np.abs(fa - want_a)) <= 1e-10 * scale
    assert np.max(np.abs(fb - want_b)) <= 1e-10 * scale


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["cfg_ethane.npz", "cfg_cn_chain.npz"])
def test_uhf_reduces_to_rhf(name):
    case = Case.load_npz(GOLD / name)
    h = liberi.Handle()
    h.setup(case.basis)
    f = h.fock_build(case.density)
    half = 0.5 * case.density
    fa, fb = h.fock_build_uhf(half, half)
    # an RHF build after the UHF one still uses its own (graph) path
    f2 = h.fock_build(case.density)
    h.destroy()
    scale = max(1.0, float(np.max(np.abs(f))))
    for g in (fa, fb, f2):
        assert np.max(np.abs(g - f)) <= 1e-11 * scale


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["cfg_water.npz", "cfg_ethane.npz"])
def test_uhf_graph_matches_builds_one_after_the_other(name):
    """From the second call on the same arrays both spins' builds run side by
    side from one graph: every replay equals the eager builds to summation
    order (1e-12 of the largest element), with other densities in the arrays,
    with restricted builds in between, on other arrays, and after a return to
    eager builds."""
    case = Case.load_npz(GOLD / name)
    rng = np.random.default_rng(5)
    b = case.basis
    pairs = [(0.5 * case.density, 0.5 * rng.permutation(case.density)), (0.7 * case.density, 0.1 * case.density)]
    h = liberi.Handle()
    h.setup(b)
    h.set_option(liberi.OPT_GRAPH, 0)
    want = [[f.copy() for f in h.fock_build_uhf(*p)] for p in pairs]
    rhf = h.fock_build(case.density).copy()
    h.set_option(liberi.OPT_GRAPH, 1)
    for call in range(6):
        got = h.fock_build_uhf(*pairs[call % 2])
        for g, w in zip(got, want[call % 2]):
            assert np.max(np.abs(g - w)) <= 1e-12 * max(1.0, float(np.max(np.abs(w))))
        if call == 3:
            assert np.max(np.abs(h.fock_build(case.density) - rhf)) <= 1e-12 * max(1.0, float(np.max(np.abs(rhf))))
    h.setup(b)  # a new setup drops the graph
    got = h.fock_build_uhf(*pairs[1])
    assert np.max(np.abs(got[0] - want[1][0])) <= 1e-12 * max(1.0, float(np.max(np.abs(want[1][0]))))
    h.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["cfg_water.npz", "cfg_ethane.npz", "cfg_cn_chain.npz"])
def test_unrestricted_builds_on_device_arrays_and_streams(name):
    """Unrestricted builds on two sets of device arrays, A on one stream and B
    on another, with a restricted build among them and nothing waited for
    on the host: first calls, calls that capture the graph of both spins, replays,
    and an eager one at the end.  Each equals the build of a handle of its own
    without graphs, to summation order (1e-12 of the largest element)."""
    from gms_liberi_amd import hipmem

    case = Case.load_npz(GOLD / name)
    n = case.basis.ntri
    rng = np.random.default_rng(6)
    dens = {"A": (0.6 * case.density, 0.5 * rng.permutation(case.density)), "B": (0.3 * case.density, 0.9 * case.density)}
    ref = liberi.Handle()
    ref.set_option(liberi.OPT_GRAPH, 0)
    ref.setup(case.basis)
    want = {k: [f.copy() for f in ref.fock_build_uhf(*d)] for k, d in dens.items()}
    want["R"] = [ref.fock_build(case.density).copy()]
    ref.destroy()

    h = liberi.Handle()
    h.setup(case.basis)
    arrays = {k: [hipmem.DeviceArray.from_host(x) for x in d] + [hipmem.DeviceArray(n), hipmem.DeviceArray(n)]
              for k, d in dens.items()}
    arrays["R"] = [hipmem.DeviceArray.from_host(case.density), hipmem.DeviceArray(n)]
    streams = [hipmem.Stream(), hipmem.Stream()]
    got = []

    def build(k, s):
        a = arrays[k]
        if k == "R":
            h.fock_build_device(a[0].address, a[1].address, n, s.address)
        else:
            assert h._lib.liberi_c_fock_build_uhf_device(h._h, *[x.ptr for x in a], n, s.ptr) == 0
        for f, w in zip(a[len(a) // 2:], want[k]):
            p = hipmem.PinnedArray(n)
            f.copy_to_async(p, s)
            got.append((k, p, w))

    for k in "AABBAARBAB":
        build(k, streams[k != "A"])
    for s in streams:
        s.synchronize()
    h.set_option(liberi.OPT_GRAPH, 0)
    build("A", streams[1])
    streams[1].synchronize()
    for i, (k, p, w) in enumerate(got):
        assert np.max(np.abs(p.array - w)) <= 1e-12 * max(1.0, float(np.max(np.abs(w)))), (i, k)
    h.destroy()
    for s in streams:
        s.destroy()
