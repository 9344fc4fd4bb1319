"""Handle lifecycle, error behaviour and rank splitting of the HIP library (GPU).

Error behaviour follows the reference: a Fock build before setup is an error
(src/interface/liberi_interface.F90:219-222); the GAMESS wrapper rejects a
build before liberi_init and a wrong matrix size
(src/interface/gms_liberi_wrapper.F90:117-127); setup on a set-up handle
cleans up first (liberi_interface.F90:133-136).
"""
import json
from pathlib import Path

import numpy as np
import pytest

from gms_liberi_amd import liberi
from gms_liberi_amd.caseio import Case
from tests.test_oracle import screening_basis

GOLD = Path(__file__).resolve().parent / "golden"


@pytest.mark.gpu
def test_build_before_setup_is_an_error():
    h = liberi.Handle()
    with pytest.raises(liberi.LiberiError) as e:
        h.fock_build(np.zeros(10))
    assert e.value.code == 2
    h.destroy()


@pytest.mark.gpu
def test_wrong_size_and_resetup():
    case = Case.load_npz(GOLD / "cfg_water.npz")
    h = liberi.Handle()
    h.setup(case.basis)
    with pytest.raises(liberi.LiberiError) as e:
        h.fock_build(np.zeros(case.basis.ntri + 1))
    assert e.value.code == 3
    f1 = h.fock_build(case.density)
    h.setup(case.basis)  # implicit cleanup
    f2 = h.fock_build(case.density)
    assert np.max(np.abs(f1 - f2)) <= 1e-12
    h.cleanup()
    with pytest.raises(liberi.LiberiError):
        h.fock_build(case.density)
    h.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["cfg_ethane", "cfg_cn_chain"])
def test_primitive_pair_screen_is_below_summation_noise(name):
    """Primitive pairs dropped at setup (their bound times the largest bound
    among the shell pairs they can meet through the quartet test is below the
    cutoff) move F by no more than summation-order noise: within 1e-12 of the
    largest element of the build that keeps every primitive pair; quartet
    counts are the same."""
    case = Case.load_npz(GOLD / f"{name}.npz")
    h0 = liberi.Handle()
    h0.set_option(liberi.OPT_PRIM_CUTOFF, 0.0)
    h0.setup(case.basis)
    f0 = h0.fock_build(case.density)
    st0 = h0.stats()
    h0.destroy()
    h = liberi.Handle()
    assert h.get_option(liberi.OPT_PRIM_CUTOFF) == 1e-18
    h.setup(case.basis)
    f = h.fock_build(case.density)
    st = h.stats()
    h.destroy()
    assert st0["prim_pairs_dropped"] == 0
    assert np.array_equal(st["quartets"], st0["quartets"])
    assert st["prim_pairs"] + st["prim_pairs_dropped"] == st0["prim_pairs"]
    if name == "cfg_cn_chain":
        assert st["prim_pairs_dropped"] > 0
    scale = max(1.0, float(np.max(np.abs(f0))))
    assert np.max(np.abs(f - f0)) <= 1e-12 * scale


@pytest.mark.gpu
def test_setup_failing_part_way_leaves_a_reusable_handle(oracle):
    """A setup that runs out of its device budget after some classes are set
    up (LIBERI_OPT_MAX_DEVICE_BYTES) fails with ENOMEM and releases everything
    it allocated; the same handle then sets up a smaller basis whose classes
    are a subset of the failed one's, and builds it exactly as a fresh handle
    and the oracle do."""
    big = Case.load_npz(GOLD / "cfg_ethane.npz")
    small = Case.load_npz(GOLD / "ref_h2o_ccpvdz.npz")
    probe = liberi.Handle()
    probe.setup(big.basis)
    full = probe.stats()["device_bytes"]
    probe.destroy()
    h = liberi.Handle()
    for frac in (0.5, 0.9):
        h.set_option(liberi.OPT_MAX_DEVICE_BYTES, frac * full)
        with pytest.raises(liberi.LiberiError) as e:
            h.setup(big.basis)
        assert e.value.code == 5 and "budget" in str(e.value)
        assert h.stats()["device_bytes"] == 0
        assert h.stats()["total_quartets"] == 0
        with pytest.raises(liberi.LiberiError) as e:  # not set up
            h.fock_build(big.density)
        assert e.value.code == 2
    h.set_option(liberi.OPT_MAX_DEVICE_BYTES, 0.0)
    h.setup(small.basis)
    f = h.fock_build(small.density)
    st = h.stats()
    h.destroy()
    f_or, counts, _ = oracle.fock(small.basis, small.density)
    assert np.max(np.abs(f - f_or)) <= 1e-10
    assert np.max(np.abs(f - small.fock)) <= 1e-10
    assert np.array_equal(st["quartets"], counts)


@pytest.mark.gpu
def test_basis_beyond_32_bit_packed_size_is_rejected():
    """num_bas(num_bas+1)/2 is a default integer in the reference's interface;
    the kernels index packed matrices in 32 bits, so setup refuses
    num_bas > 65535 with an argument error before touching the arrays."""
    import dataclasses

    b = Case.load_npz(GOLD / "cfg_water.npz").basis
    h = liberi.Handle()
    with pytest.raises(liberi.LiberiError) as e:
        h.setup(dataclasses.replace(b, num_bas=65536))
    assert e.value.code == 1
    h.destroy()


@pytest.mark.gpu
def test_gamess_wrapper_entry_points():
    case = Case.load_npz(GOLD / "ref_h2o_ccpvdz.npz")
    b = case.basis
    f = np.zeros(b.ntri)
    with pytest.raises(liberi.LiberiError) as e:
        liberi.liberi_fock(case.density, f, b.ntri)
    assert e.value.code == 2
    liberi.liberi_init(b.natoms, b.num_bas, b.nsh, b.mxgtot, b.ang_mom, b.contr_num, b.sh_loc, b.atom_num,
                       b.atom_loc, b.start_bas, b.end_bas, b.exponents, b.coef_s, b.coef_p, b.coef_d, b.coef_f,
                       b.coords, b.schwrz, 0, 1)
    with pytest.raises(liberi.LiberiError) as e:
        liberi.liberi_fock(case.density, f, b.ntri - 1)
    assert e.value.code == 3
    liberi.liberi_fock(case.density, f, b.ntri)
    assert np.max(np.abs(f - case.fock)) <= 1e-10
    liberi.liberi_finalize()


@pytest.mark.gpu
def test_reference_named_functions():
    case = Case.load_npz(GOLD / "ref_h2_ccpvdz.npz")
    b = case.basis
    h = liberi.liberi_create()
    liberi.liberi_setup(h, b.nsh, b.natoms, b.num_bas, b.mxgtot, b.ang_mom, b.contr_num, b.sh_loc, b.atom_num,
                        b.atom_loc, b.start_bas, b.end_bas, b.exponents, b.coef_s, b.coef_p, b.coef_d, b.coef_f,
                        b.coords, b.schwrz, 0, 1)
    f = np.full(b.ntri, 7.0)  # overwritten, not accumulated (src/liberi_driver.F90:64)
    liberi.liberi_fock_build(h, case.density, f, b.ntri)
    assert np.max(np.abs(f - case.fock)) <= 1e-10
    liberi.liberi_cleanup(h)
    liberi.liberi_destroy(h)


@pytest.mark.gpu
@pytest.mark.parametrize("split", [0, 1])
@pytest.mark.parametrize("nprocs", [2, 3, 8])
def test_rank_partials_sum_to_full(nprocs, split):
    """Each rank returns its partial F; the caller's sum is the full F, for the
    cost-balanced shares (split 0) and the reference's equal counts (split 1);
    the shares' quartets and primitive quartets add up to the class totals."""
    case = Case.load_npz(GOLD / "cfg_ethane.npz")
    h = liberi.Handle()
    h.set_option(liberi.OPT_RANK_SPLIT, split)
    h.setup(case.basis)
    full = h.fock_build(case.density)
    total_q = h.stats()["quartets"].copy()
    total_pq = h.stats()["prim_quartets"].copy()
    acc = np.zeros_like(full)
    q = np.zeros_like(total_q)
    pq = np.zeros_like(total_pq)
    for r in range(nprocs):
        h.setup(case.basis, my_rank=r, num_procs=nprocs)
        acc += h.fock_build(case.density)
        q += h.stats()["quartets"]
        pq += h.stats()["prim_quartets"]
        if split == 1:  # the reference's split: equal counts, the last rank the remainder
            assert np.all(np.abs(h.stats()["quartets"] - total_q / nprocs) <= 1)
    h.destroy()
    assert np.array_equal(q, total_q) and np.array_equal(pq, total_pq)
    assert np.max(np.abs(acc - full)) <= 1e-12


@pytest.mark.gpu
def test_screening_counts_reference_targets():
    d = json.loads((GOLD / "ref_screening_w2_631gd.json").read_text())
    h = liberi.Handle()
    h.setup(screening_basis(d))
    counts = h.stats()["quartets"]
    h.destroy()
    names = liberi.class_names()
    assert [int(counts[names.index(k)]) for k in d["classes"]] == d["alternative_target"]


@pytest.mark.gpu
def test_device_resident_build_matches_host_build():
    from gms_liberi_amd import hipmem

    case = Case.load_npz(GOLD / "cfg_ethane.npz")
    h = liberi.Handle()
    h.setup(case.basis)
    host = h.fock_build(case.density)
    D = hipmem.DeviceArray.from_host(case.density)
    F = hipmem.DeviceArray.from_host(np.full(case.basis.ntri, 3.0))
    s = hipmem.Stream()
    h.fock_build_device(D.address, F.address, case.basis.ntri, s.address)
    s.synchronize()
    got = F.to_host()
    h.destroy()
    s.destroy()
    assert np.max(np.abs(got - host)) <= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["ref_h2o_ccpvtz.npz", "cfg_ethane.npz"])
def test_exact_large_t_mode_matches_oracle(name, oracle):
    """With the large-argument switch moved to where it is exact, the build
    agrees with the independent McMurchie-Davidson oracle."""
    case = Case.load_npz(GOLD / name)
    h = liberi.Handle()
    h.set_option(liberi.OPT_EXACT_LARGE_T, 1)
    h.setup(case.basis)
    f = h.fock_build(case.density)
    h.destroy()
    fo, _, _ = oracle.fock(case.basis, case.density)
    assert np.max(np.abs(f - fo)) <= 1e-11 * max(1.0, np.max(np.abs(fo)))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["cfg_ethane.npz", "cfg_cn_chain.npz"])
def test_row_tiles_match_direct_digestion(name):
    """Row-tiled digestion (exchange blocks of a tile's fixed pair accumulated
    on chip, in either orientation) and per-quartet atomic digestion give the
    same F up to summation order."""
    case = Case.load_npz(GOLD / name)
    h = liberi.Handle()
    h.setup(case.basis)
    assert h.get_option(liberi.OPT_ROW_TILES) == 1.0
    h.set_option(liberi.OPT_ROW_TILES, 2)
    tiled = h.fock_build(case.density)
    variants = h.stats()["class_variant"]
    h.set_option(liberi.OPT_ROW_TILES, 0)
    direct = h.fock_build(case.density)
    # no row tiles left; the f classes keep their timed group/cooperative form
    assert np.all(np.isin(h.stats()["class_variant"][variants >= 0], [0, 3]))
    h.destroy()
    assert np.any(variants == 1) and np.any(variants == 2)  # both orientations ran
    scale = max(1.0, float(np.max(np.abs(direct))))
    assert np.max(np.abs(tiled - direct)) <= 1e-11 * scale
    # against the reference's own F: 1e-10, except where the reference's
    # (sp|dd) kernel is itself inexact (the C-N chain, see test_gpu_parity)
    assert np.max(np.abs(tiled - case.fock)) <= (1e-9 if "chain" in name else 1e-10)


@pytest.mark.gpu
def test_autotuned_build_matches_reference():
    """The first build times both digestion forms per class and keeps the
    faster; every later build uses the choice.  F is the same either way."""
    case = Case.load_npz(GOLD / "cfg_cn_chain.npz")
    h = liberi.Handle()
    h.setup(case.basis)
    assert np.all(h.stats()["class_variant"] == -1)  # nothing chosen before the first build
    f1 = h.fock_build(case.density)
    v1 = h.stats()["class_variant"].copy()
    f2 = h.fock_build(case.density)
    v2 = h.stats()["class_variant"].copy()
    h.set_option(liberi.OPT_AUTOTUNE, 0)
    f3 = h.fock_build(case.density)
    v3 = h.stats()["class_variant"].copy()
    h.destroy()
    active = v1 >= 0
    assert active.sum() > 20 and np.array_equal(v1, v2)
    assert np.array_equal(v3 >= 0, active)
    # untimed: the group form for every f class that also has the cooperative
    # one; (ff|dd), (ff|fd) and (ff|ff) have only the cooperative form
    names = liberi.class_names()
    coop_only = np.array([n in ("int3322", "int3332", "int3333") for n in names])
    assert np.array_equal(v3 == 3, coop_only & active)
    assert np.all(v1[coop_only & active] == 3)
    print("cooperative form chosen for", [liberi.class_names()[c] for c in np.flatnonzero(v1 == 3)])
    # the forms differ only in the order of the FP64 additions into F: within
    # 1e-13 of the largest element (elements of the chain reach ~1.3e3)
    scale = max(1.0, float(np.max(np.abs(f1))))
    for f in (f1, f2, f3):
        assert np.max(np.abs(f - f1)) <= 1e-13 * scale
    dE = 0.5 * float(np.dot(case.density, f1 - case.fock))
    assert abs(dE) <= 1e-9


@pytest.mark.gpu
def test_graph_replays_match_eager_builds():
    """Batched form: class launches on four side streams captured into one HIP
    graph.  Every replay, with eager work and synchronisations in between and
    a new density in the same buffer, equals the eager build."""
    from gms_liberi_amd import hipmem

    case = Case.load_npz(GOLD / "cfg_ethane.npz")
    rng = np.random.default_rng(4)
    dens = [case.density, case.density * (1.0 + 0.01 * rng.standard_normal(case.density.shape))]
    h = liberi.Handle()
    h.setup(case.basis)
    assert h.get_option(liberi.OPT_GRAPH) == 1.0
    h.set_option(liberi.OPT_GRAPH, 0)
    eager = [h.fock_build(d) for d in dens]
    h.set_option(liberi.OPT_GRAPH, 1)
    n = case.basis.ntri
    D = hipmem.DeviceArray(n)
    F = hipmem.DeviceArray(n)
    s = hipmem.Stream()
    for rep in range(4):
        k = rep % 2
        D.copy_from_async(_pinned(dens[k]), s)
        h.fock_build_device(D.address, F.address, n, s.address)
        s.synchronize()
        got = F.to_host()
        assert np.max(np.abs(got - eager[k])) <= 1e-12, rep
        assert np.max(np.abs(h.fock_build(dens[k]) - eager[k])) <= 1e-12  # host path, its own graph
    h.destroy()
    s.destroy()


def _pinned(a):
    from gms_liberi_amd import hipmem

    p = hipmem.PinnedArray(a.shape[0])
    p.array[:] = a
    _pinned.keep.append(p)
    return p


_pinned.keep = []


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["cfg_ethane.npz", "cfg_cn_chain.npz", "cfg_c60.npz"])
def test_fused_group_launch_matches_per_class_launches(name):
    """LIBERI_OPT_FUSED: the s, p, d group classes in one persistent launch fed
    from a device work queue give the per-class launches' Fock matrix (to
    summation order), graph-captured and replayed as well as eager."""
    case = Case.load_npz(GOLD / name)
    out = {}
    for fused in (0, 1):
        for graph in (0, 1):
            h = liberi.Handle()
            h.set_option(liberi.OPT_FUSED, fused)
            h.set_option(liberi.OPT_GRAPH, graph)
            h.setup(case.basis)
            f = [h.fock_build(case.density) for _ in range(3)]
            v = h.stats()["class_variant"]
            h.destroy()
            assert np.any(v == 4) == bool(fused)  # every case has fused classes
            out[(fused, graph)] = f
    ref = out[(0, 0)][0]
    scale = max(1.0, float(np.max(np.abs(ref))))
    for k, fs in out.items():
        for f in fs:
            assert np.max(np.abs(f - ref)) <= 1e-11 * scale, k


@pytest.mark.gpu
def test_row_tile_lengths_give_the_same_fock():
    """Every row-tile length (LIBERI_OPT_TILE_LEN) and the per-class timed
    choice give the reference's Fock matrix, equal to summation order; the
    statistics report the length each row-tiled class ran with."""
    case = Case.load_npz(GOLD / "cfg_c60.npz")
    h = liberi.Handle()
    h.setup(case.basis)
    out = {}
    for length in (0, 512, 1024, 4096, 16384):
        h.set_option(liberi.OPT_TILE_LEN, length)
        assert h.get_option(liberi.OPT_TILE_LEN) == length
        out[length] = h.fock_build(case.density)
        st = h.stats()
        row = (st["class_variant"] == 1) | (st["class_variant"] == 2)
        assert row.sum() >= 10
        assert np.all(st["class_tile"][~row] == 0)
        if length:
            assert np.all(st["class_tile"][row] == length)
        else:
            assert set(st["class_tile"][row].tolist()) <= {512, 1024, 4096, 16384}
            print("tile lengths chosen:", {liberi.class_names()[c]: int(st["class_tile"][c])
                                           for c in np.flatnonzero(row)})
    with pytest.raises(liberi.LiberiError):
        h.set_option(liberi.OPT_TILE_LEN, 2048)
    h.destroy()
    scale = max(1.0, float(np.max(np.abs(out[0]))))
    for length, f in out.items():
        assert np.max(np.abs(f - out[0])) <= 1e-13 * scale, length
    # F against the reference class by class: test_gpu_parity
    assert abs(0.5 * float(np.dot(case.density, out[0] - case.fock))) <= 1e-9


SPLIT_CLASSES = ["int2120", "int2220", "int0122", "int2111", "int2121", "int2221", "int2211",
                 "int2130", "int2230", "int3120", "int3130", "int3111", "int3121", "int2231", "int3131"]
SPLIT_DIAGONAL = ["int2121", "int3131"]


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["cfg_ethane.npz", "cfg_cn_chain.npz", "cfg_c60.npz"])
def test_wave_split_forms_match_group_forms(name):
    """The wave-split row-tiled form of the d and f classes -- slices of (e0|f0)
    (columns, rows, or the cone of one C component) held in registers by the
    waves of a workgroup, exchange rows in LDS -- in both orientations of the
    row tiles, equals the group form with direct atomics, class by class."""
    case = Case.load_npz(GOLD / name)
    names = liberi.class_names()
    for orient in (1, 2):
        h = liberi.Handle()
        h.set_option(liberi.OPT_ROW_ORIENT, orient)
        h.setup(case.basis)
        counts = h.stats()["quartets"]
        for k in SPLIT_CLASSES:
            c = names.index(k)
            if counts[c] == 0:
                continue
            h.set_option(liberi.OPT_ONLY_CLASS, c)
            h.set_option(liberi.OPT_ROW_TILES, 2)
            split = h.fock_build(case.density)
            variant = int(h.stats()["class_variant"][c])
            h.set_option(liberi.OPT_ROW_TILES, 0)
            direct = h.fock_build(case.density)
            assert int(h.stats()["class_variant"][c]) in (0, 3)  # group or cooperative form
            diag = k in SPLIT_DIAGONAL
            err = float(np.max(np.abs(split - direct)))
            print(f"{name} orient {orient} {k}: variant {variant}, max|split - group| {err:.2e}", flush=True)
            assert variant == (1 if diag else orient)
            assert err <= 1e-12 * max(1.0, float(np.max(np.abs(direct))))
        h.destroy()


@pytest.mark.gpu
def test_untimed_first_build_captured_in_a_graph():
    """With the autotuner off, the first build after setup is captured straight
    into the graph: the wave-split kernels (their LDS limit raised at handle
    creation, outside any capture) run from it, and every replay equals the
    reference."""
    from gms_liberi_amd import hipmem

    case = Case.load_npz(GOLD / "cfg_ethane.npz")
    names = liberi.class_names()
    h = liberi.Handle()
    h.set_option(liberi.OPT_AUTOTUNE, 0)
    h.setup(case.basis)
    n = case.basis.ntri
    D = hipmem.DeviceArray.from_host(case.density)
    F = hipmem.DeviceArray(n)
    s = hipmem.Stream()
    for _ in range(3):
        h.fock_build_device(D.address, F.address, n, s.address)
        s.synchronize()
        assert np.max(np.abs(F.to_host() - case.fock)) <= 1e-10
    variants = h.stats()["class_variant"]
    counts = h.stats()["quartets"]
    assert all(variants[names.index(k)] in (1, 2) for k in SPLIT_CLASSES if counts[names.index(k)] > 0)
    h.destroy()
    s.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("mol,natoms,ranks", [("water", 3, 1), ("ethane", 8, 1), ("cn_chain", 2, 1), ("cn_chain", 3, 3),
                                              ("cn_chain", 5, 1), ("cluster", 9, 4), ("cage", 7, 1), ("cage", 12, 8)])
def test_shared_launches_match_launches_per_class(mol, natoms, ranks):
    """Small classes run several to a launch, each workgroup its class's body:
    the same F as launches of one class (no tuning: none is shared), replayed
    from a graph and launched eagerly, for classes from one quartet to those
    that no longer share, and for shares of a build.  The forms differ in the
    order of the FP64 additions: 1e-12 of the largest element."""
    from gms_liberi_amd import configs

    case = {"water": lambda: configs.water(3), "ethane": lambda: configs.ethane(4),
            "cn_chain": lambda: configs.cn_chain(5, natoms), "cluster": lambda: configs.cluster(natoms, 6),
            "cage": lambda: configs.c60_fragment(natoms, 7)}[mol]()
    b = case.basis.with_schwarz(liberi.schwarz(case.basis))
    total = {}
    for rank in range(ranks):
        h = liberi.Handle()
        h.setup(b, rank, ranks)
        got = [("shared", h.fock_build(case.density).copy()), ("shared", h.fock_build(case.density).copy())]
        h.set_option(liberi.OPT_GRAPH, 0)
        got.append(("shared", h.fock_build(case.density).copy()))
        h.set_option(liberi.OPT_AUTOTUNE, 0)
        got.append(("single", h.fock_build(case.density).copy()))
        h.destroy()
        scale = max(1.0, float(np.max(np.abs(got[-1][1]))))
        for _, f in got:
            assert np.max(np.abs(f - got[-1][1])) <= 1e-12 * scale
        total["shared"] = total.get("shared", 0) + got[0][1]
    h = liberi.Handle()
    h.setup(b)
    h.set_option(liberi.OPT_AUTOTUNE, 0)
    whole = h.fock_build(case.density)
    h.destroy()
    assert np.max(np.abs(total["shared"] - whole)) <= 1e-12 * max(1.0, float(np.max(np.abs(whole))))


@pytest.mark.gpu
@pytest.mark.parametrize("name,graph", [("cfg_water.npz", 1), ("cfg_ethane.npz", 1), ("cfg_ethane.npz", 0),
                                        ("cfg_cn_chain.npz", 1)])
def test_builds_in_graphs_of_the_callers(name, graph):
    """Two builds of one handle captured by the caller, each into its own graph
    and Fock array, replayed side by side and beside the handle's own builds on
    a third stream: each replay equals the eager build of its density to
    summation order (1e-12 of the largest element), over several replays with
    new densities."""
    import ctypes as C

    from gms_liberi_amd import hipmem

    case = Case.load_npz(GOLD / name)
    n = case.basis.ntri
    rng = np.random.default_rng(3)
    ref = liberi.Handle()
    ref.set_option(liberi.OPT_GRAPH, 0)
    ref.setup(case.basis)
    h = liberi.Handle()
    h.set_option(liberi.OPT_GRAPH, graph)
    h.setup(case.basis)
    rt = hipmem.runtime()
    streams = [hipmem.Stream() for _ in range(3)]
    D = [hipmem.DeviceArray.from_host(case.density) for _ in range(3)]
    F = [hipmem.DeviceArray(n) for _ in range(3)]
    h.fock_build_device(D[2].address, F[2].address, n, streams[2].address)
    execs = []
    for k in range(2):
        s, g, e = streams[k], C.c_void_p(), C.c_void_p()
        assert rt.hipStreamBeginCapture(s.ptr, 2 * k) == 0  # global and relaxed mode
        h.fock_build_device(D[k].address, F[k].address, n, s.address)
        assert rt.hipStreamEndCapture(s.ptr, C.byref(g)) == 0
        assert rt.hipGraphInstantiate(C.byref(e), g, None, None, C.c_size_t(0)) == 0
        assert rt.hipGraphDestroy(g) == 0
        execs.append(e)
    h.fock_build_device(D[2].address, F[2].address, n, streams[2].address)
    streams[2].synchronize()
    for step in range(4):
        dens = [np.ascontiguousarray(x * case.density) for x in rng.uniform(0.2, 1.0, 3)]
        for d, a in zip(dens, D):
            assert rt.hipMemcpy(a.ptr, d.ctypes.data, d.nbytes, 1) == 0
        for _ in range(3):  # (nothing waited for between them)
            for k in range(2):
                assert rt.hipGraphLaunch(execs[k], streams[k].ptr) == 0
            h.fock_build_device(D[2].address, F[2].address, n, streams[2].address)
        for s in streams:
            s.synchronize()
        for k in range(3):
            want = ref.fock_build(dens[k])
            assert np.max(np.abs(F[k].to_host() - want)) <= 1e-12 * max(1.0, float(np.max(np.abs(want)))), (step, k)
    for e in execs:
        assert rt.hipGraphExecDestroy(e) == 0
    h.destroy()
    ref.destroy()
    for s in streams:
        s.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("natoms", [5, 17])
def test_asked_tile_lengths_in_small_classes(natoms):
    """LIBERI_OPT_TILE_LEN in classes of few quartets, which run one workgroup
    step a tile where none is asked for: the same Fock matrix to summation order
    (1e-12 of the largest element), and the statistics give the length."""
    from gms_liberi_amd import configs

    case = configs.cluster(natoms, 5)
    h = liberi.Handle()
    h.setup(case.basis.with_schwarz(liberi.schwarz(case.basis)))
    ref = h.fock_build(case.density).copy()
    for length in (512, 1024, 4096, 16384, 0):
        h.set_option(liberi.OPT_TILE_LEN, length)
        f = h.fock_build(case.density)
        assert np.max(np.abs(f - ref)) <= 1e-12 * max(1.0, float(np.max(np.abs(ref)))), length
        st = h.stats()
        row = (st["class_variant"] == 1) | (st["class_variant"] == 2)
        assert row.any() and np.all(st["class_tile"][~row] == 0)
        if length:
            assert np.all(st["class_tile"][row] == length)
        else:
            assert np.all(st["class_tile"][row] <= 512)
    h.destroy()
