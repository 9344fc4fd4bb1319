"""What the host code of the built library allocates, launches, orders and
frees, on the HIP calls of hip_host.cpp in place of the runtime (no GPU).

Each scenario runs in a process of its own, in which those calls come before
the runtime's."""
import ctypes as C
import re
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


@pytest.fixture(scope="session")
def host_lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("hip_host") / "hip_host.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-I/opt/rocm/include", "-o", str(so),
                    str(ROOT / "tests" / "hip_host.cpp"), "-ldl"], check=True)
    return so


def run(scenario, host_lib):
    p = subprocess.run([sys.executable, __file__, str(host_lib), scenario], capture_output=True, text=True, timeout=300,
                       cwd=ROOT)
    assert p.returncode == 0, f"{scenario}: exit {p.returncode}\n{p.stdout[-2000:]}\n{p.stderr[-4000:]}"


class Host:
    """The calls of hip_host.cpp, loaded before the library."""

    def __init__(self, so):
        self.c = C.CDLL(so, C.RTLD_GLOBAL)
        self.c.host_log.restype = C.c_char_p
        for f in ("host_bytes", "host_peak"):
            getattr(self.c, f).restype = C.c_size_t
        self.c.host_fail.argtypes = [C.c_size_t]
        vp = C.c_void_p
        for f in ("host_id", "host_in_flight", "host_outstanding"):
            getattr(self.c, f).argtypes = [vp]
        self.c.host_outstanding.restype = C.c_long
        self.c.host_before.argtypes = [vp, vp]
        self.c.hipStreamBeginCapture.argtypes = [vp, C.c_int]
        self.c.hipStreamEndCapture.argtypes = [vp, C.POINTER(vp)]

    def stream(self):
        s = C.c_void_p()
        assert self.c.hipStreamCreateWithFlags(C.byref(s), 0) == 0
        return s

    def array(self, values):
        """A device array (host memory here)."""
        values = np.ascontiguousarray(values, dtype=np.float64)
        p = C.c_void_p()
        assert self.c.hipMalloc(C.byref(p), C.c_size_t(values.nbytes)) == 0
        C.memmove(p, values.ctypes.data, values.nbytes)
        return p

    def begin_capture(self, s):
        assert self.c.hipStreamBeginCapture(s, 0) == 0

    def end_capture(self, s):
        g = C.c_void_p()
        assert self.c.hipStreamEndCapture(s, C.byref(g)) == 0

    def log(self):
        """The lines since the last call."""
        lines = self.c.host_log().decode().splitlines()
        self.c.host_clear()
        return lines


def field(line, name):
    m = re.search(rf"\b{name}=(\S+)", line)
    return m and (int(m.group(1)) if m.group(1).isdigit() else m.group(1))


def golden(name):
    from gms_liberi_amd.caseio import Case

    return Case.load_npz(ROOT / "tests" / "golden" / name).basis


def row_of_s(n, spacing=1.4):
    """n atoms in a row, one tight s primitive each; Schwarz values of 1 keep
    every pair, and most pairs have no primitive pair left (at 1.4 bohr)."""
    from gms_liberi_amd.caseio import Basis

    one = np.arange(n) + 1
    coef = np.zeros((4, n))
    coef[0] = 1.0
    xyz = np.zeros((n, 3))
    xyz[:, 0] = spacing * np.arange(n)
    return Basis(n, n, n, 1, np.ones(n, int), np.ones(n, int), one, one, one, one, one, np.full(n, 3.4), *coef, xyz.ravel(),
                 np.ones(n * (n + 1) // 2))


# ------------------------------------------------------------- scenarios
def scenario_pairs_without_primitives(host):
    """A kernel may read the first record of any pair it is given: those of a
    pair without primitives lie inside the array as well."""
    from gms_liberi_amd import liberi

    h = liberi.Handle()
    h.setup(row_of_s(100))
    h.fock_build(np.zeros(100 * 101 // 2))
    begin = [x for x in host.log() if "build_begin" in x]
    assert begin and field(begin[0], "empty") > 3000
    assert field(begin[0], "past") == 0, begin[0]
    h.destroy()


def scenario_builds_on_other_streams_wait(host):
    """Every build of a handle comes after the last one that runs, whatever
    its stream, restricted or not, also where one was captured in between."""
    from gms_liberi_amd import liberi

    b = golden("cfg_water.npz")
    n = b.ntri
    streams = [host.stream() for _ in range(4)]
    D, F, Da, Db, Fa, Fb = (host.array(np.zeros(n)) for _ in range(6))
    h = liberi.Handle()
    h.setup(b)

    def rhf(s):
        h.fock_build_device(D.value, F.value, n, s.value)

    def uhf(s):
        assert h._lib.liberi_c_fock_build_uhf_device(h._h, Da, Db, Fa, Fb, n, s) == 0

    uhf(streams[0])
    for first in (rhf, uhf):
        for second in (rhf, uhf):
            for captured in (None, rhf, uhf):
                a, x, c, d = streams
                first(a)
                if captured:
                    host.begin_capture(x)
                    captured(x)
                    host.end_capture(x)
                second(c)
                assert host.c.host_before(a, c), (first.__name__, captured and captured.__name__, second.__name__)
                second(d)  # (the unrestricted graph from its second call on)
                assert host.c.host_before(c, d)
    assert h.stats()["last_build_ms"] > 0
    h.destroy()


def scenario_unrestricted_builds_without_a_second_workspace(host):
    """Where the second workspace of the side-by-side unrestricted build is
    refused, by the device or by the handle's budget, the builds run one
    after the other; it is asked for once."""
    from gms_liberi_amd import liberi

    b = golden("cfg_water.npz")
    n = b.ntri
    s = host.stream()
    arrays = [host.array(np.zeros(n)) for _ in range(4)]

    def build(h):
        host.log()
        rc = h._lib.liberi_c_fock_build_uhf_device(h._h, *arrays, n, s)
        return rc, host.log()

    h = liberi.Handle()
    h.setup(b)
    assert build(h)[0] == 0
    rc, lines = build(h)
    size = [field(x.replace("malloc ", "malloc="), "malloc") for x in lines if x.startswith("malloc")]
    assert rc == 0 and len(size) == 1 and any("replay" in x for x in lines)
    with pytest.raises(liberi.LiberiError):
        h.fock_build(np.zeros(n + 1))
    message = h._lib.liberi_c_last_error()
    h.destroy()
    for budgeted in (False, True):
        h = liberi.Handle()
        h.setup(b)
        assert build(h)[0] == 0
        h.set_option(liberi.OPT_MAX_DEVICE_BYTES, h.stats()["device_bytes"] + size[0] - 1 if budgeted else 0)
        host.c.host_fail(0 if budgeted else size[0])
        refused = 0
        for _ in range(3):
            rc, lines = build(h)
            assert rc == 0, h._lib.liberi_c_last_error()
            refused += sum("malloc failed" in x for x in lines)
            assert sum("build_begin" in x for x in lines) == 2 and not any("replay" in x for x in lines)
        assert refused == (0 if budgeted else 1) and h._lib.liberi_c_last_error() == message
        host.c.host_fail(0)
        h.set_option(liberi.OPT_MAX_DEVICE_BYTES, 0)  # asked for again
        assert any("replay" in x for x in build(h)[1])
        h.destroy()
    # a failed setup, or Schwarz call, leaves nothing behind for the next
    h = liberi.Handle()
    host.c.host_fail(1 << 10)
    for call in (lambda: h.setup(b), lambda: liberi.schwarz(b)):
        with pytest.raises(liberi.LiberiError) as e:
            call()
        assert e.value.code == 5
    host.c.host_fail(0)
    h.setup(b)
    h.destroy()


def scenario_graphs_end_after_their_replays(host):
    """A captured build is destroyed, whatever drops it, only after its replays
    on the caller's stream; builds on other arrays are launched before that wait."""
    from gms_liberi_amd import liberi

    b = golden("cfg_water.npz")
    n = b.ntri
    s = host.stream()
    a = [host.array(np.zeros(n)) for _ in range(4)]
    c = [host.array(np.zeros(n)) for _ in range(4)]

    def rhf(h, x):
        h.fock_build_device(x[0].value, x[1].value, n, s.value)

    def uhf(h, x):
        for _ in range(2):
            assert h._lib.liberi_c_fock_build_uhf_device(h._h, *x, n, s) == 0

    def destroyed():
        return [field(x, "in_flight") for x in host.log() if x.startswith("destroy")]

    drops = [lambda h, build: h.set_option(liberi.OPT_VALUE_CUTOFF, 1e-12), lambda h, build: h.cleanup(),
             lambda h, build: h.setup(b), lambda h, build: h.destroy(), lambda h, build: build(h, c)]
    for build in (rhf, uhf):
        for drop in drops:
            h = liberi.Handle()
            h.setup(b)
            build(h, a)
            build(h, a)
            host.log()
            assert host.c.host_in_flight(s)
            drop(h, build)
            assert destroyed() == [0], (build.__name__, drops.index(drop))
            if drop is drops[-1]:
                assert host.c.host_in_flight(s)  # the build on the other arrays
            h.destroy()
    # one that a capture of the caller's holds back
    h = liberi.Handle()
    h.setup(b)
    rhf(h, a)
    x = host.stream()
    host.begin_capture(x)
    host.log()
    h.set_option(liberi.OPT_VALUE_CUTOFF, 1e-12)
    host.end_capture(x)
    assert destroyed() == [0]
    h.destroy()


def scenario_captured_builds_have_their_own_workspace(host):
    """A build under a caller's capture (which may be replayed beside others)
    gets a workspace per Fock array, and gives it back with the handle's data."""
    from gms_liberi_amd import liberi

    b = golden("cfg_water.npz")
    n = b.ntri
    run, x = host.stream(), host.stream()
    D = host.array(np.zeros(n))
    F = [host.array(np.zeros(n)) for _ in range(3)]
    h = liberi.Handle()
    h.setup(b)
    held = h.stats()["device_bytes"]

    def build(f, s):
        host.log()
        h.fock_build_device(D.value, f.value, n, s.value)
        lines = host.log()
        assert not any("capture stream" in k or "replay" in k for k in lines) or s is run
        return {field(k, "Jp") for k in lines if "build_begin" in k}

    own = build(F[0], run)
    h.stats()
    for graph in (1, 0):
        h.set_option(liberi.OPT_GRAPH, graph)
        work = []
        host.begin_capture(x)
        for f in (F[0], F[1], F[2], F[1]):
            work.append(build(f, x))
        host.end_capture(x)
        assert all(len(w) == 1 for w in work) and work[3] == work[1]
        assert len(set.union(own, *work)) == 4
        assert build(F[0], run) <= own
    assert h.stats()["device_bytes"] > held
    before = host.c.host_bytes()
    h.cleanup()
    assert h.stats()["device_bytes"] == 0 and host.c.host_bytes() < before
    h.setup(b)
    assert h.stats()["device_bytes"] == held
    # no memory for it: refused, and the handle goes on
    h.fock_build(np.zeros(n))
    host.begin_capture(x)
    host.c.host_fail(1 << 10)
    with pytest.raises(liberi.LiberiError) as e:
        build(F[1], x)
    assert e.value.code == 5
    host.c.host_fail(0)
    host.end_capture(x)
    h.fock_build(np.zeros(n))
    h.destroy()


def launched_forms(lines):
    """Class index -> (form, longest row tile, whether shared) of a build's launches."""
    from gms_liberi_amd.census import CLASS_L

    ids = {tuple(l): k for k, l in enumerate(CLASS_L)}
    forms = {}
    for x in lines:
        m = re.search(r"eri_(small|row|split|group|coop)_kernelI((?:Li\d)+)(?:Lb([01]))?", x.replace("E", ""))
        if m:
            c = ids[tuple(int(v) for v in re.findall(r"Li(\d)", m.group(2)))]
            form = {"small": 0, "group": 0, "coop": 3}.get(m.group(1), 1 + int(m.group(3) or 0))
            forms[c] = (form, field(x, "longest") or 0, False)
        for c, tr, tiles in re.findall(r"\[class=(\d+) transposed=(\d)(.*?)\]", x):
            launch = field(x, "launch")
            forms[int(c)] = (1 + int(tr), field(tiles, "longest"), True) if launch < 3 else (0 if launch == 3 else 3, 0, True)
    return forms


def cluster(n, seed):
    from gms_liberi_amd import configs
    from tests.oracle_ctypes import Oracle

    b = configs.cluster(n, seed).basis
    return b.with_schwarz(Oracle().schwarz(b))


def scenario_statistics_name_the_launches(host):
    """class_variant and class_tile are those of the launches of the last build,
    shared or not, also after a build that chose other forms."""
    from gms_liberi_amd import liberi

    for b in (golden("cfg_ethane.npz"), golden("cfg_cn_chain.npz"), cluster(12, 21)):
        d = np.zeros(b.ntri)
        for options in ([], [(liberi.OPT_CLASS_TIMING, 1), (liberi.OPT_CLASS_TIMING, 0)], [(liberi.OPT_FP32_TAU, 1e-6)],
                        [(liberi.OPT_FP32_TAU, 1e-6), (liberi.OPT_FP32_TAU, 0)], [(liberi.OPT_ROW_TILES, 2)],
                        [(liberi.OPT_ROW_TILES, 0), (liberi.OPT_ROW_TILES, 1)], [(liberi.OPT_AUTOTUNE, 0)]):
            h = liberi.Handle()
            h.setup(b)
            assert np.all(h.stats()["class_variant"] == -1)
            for opt, value in options or [(liberi.OPT_GRAPH, 1)]:
                h.set_option(opt, value)
                h.fock_build(d)
            h.set_option(liberi.OPT_GRAPH, 0)
            host.log()
            h.fock_build(d)
            forms = launched_forms(host.log())
            st = h.stats()
            assert {c for c in range(55) if st["quartets"][c]} == set(forms)
            for c in range(55):
                form, longest, shared = forms.get(c, (-1, 0, False))
                assert st["class_variant"][c] == form, (options, c)
                assert (st["class_tile"][c] > 0) == (form in (1, 2)) and longest <= st["class_tile"][c], (options, c)
                assert not shared or st["class_tile"][c] in (256, 0), (options, c)
            h.destroy()


def scenario_forms_do_not_depend_on_when_an_option_is_set(host):
    """An option that takes classes out of their shared launch gives them the
    forms and tile lengths that they would have had from the start."""
    from gms_liberi_amd import liberi

    b = cluster(12, 21)
    d = np.zeros(b.ntri)
    for opt, value in ((liberi.OPT_FP32_TAU, 1e-6), (liberi.OPT_CLASS_TIMING, 1), (liberi.OPT_FUSED, 1),
                       (liberi.OPT_TILE_LEN, 1024), (liberi.OPT_ROW_TILES, 0), (liberi.OPT_ROW_TILES, 2)):
        seen = []
        for first in (True, False):
            h = liberi.Handle()
            h.setup(b)
            if first:
                h.fock_build(d)
            h.set_option(liberi.OPT_GRAPH, 0)
            h.set_option(opt, value)
            h.fock_build(d)
            host.log()
            h.fock_build(d)
            seen.append(sorted(re.sub(r"(stream|Jp)=\S+", "", x) for x in host.log() if x.startswith("launch")))
            liberi.Handle().set_option(liberi.OPT_AUTOTUNE, 1)  # forgets the timed choices
            h.destroy()
        assert seen[0] == seen[1], (opt, value)


def scenario_builds_under_a_capture_time_nothing(host):
    """A build under a caller's capture chooses forms without running any:
    after an option that changes them, and as the first one of a handle.  The
    next build that runs chooses as ever."""
    from gms_liberi_amd import liberi

    b = golden("cfg_ethane.npz")
    n = b.ntri
    run, x = host.stream(), host.stream()
    D, F = host.array(np.zeros(n)), host.array(np.zeros(n))

    def build(h, s):
        host.log()
        h.fock_build_device(D.value, F.value, n, s.value)
        return host.log()

    for opt, value in ((liberi.OPT_GRAPH, 0), (liberi.OPT_CLASS_TIMING, 1), (liberi.OPT_TILE_LEN, 512),
                       (liberi.OPT_ROW_TILES, 2), (liberi.OPT_ROW_TILES, 0), (liberi.OPT_FUSED, 1),
                       (liberi.OPT_FP32_TAU, 1e-6), (liberi.OPT_AUTOTUNE, 0), (liberi.OPT_AUTOTUNE, 1)):
        for first in (True, False):
            h = liberi.Handle()
            h.setup(b)
            if first:
                build(h, run)
            h.set_option(opt, value)
            host.begin_capture(x)
            captured = build(h, x)
            host.end_capture(x)
            assert all(field(k, "captured") == 1 for k in captured if k.startswith("launch"))
            counts = h.stats()["quartets"]
            assert sum(v in launched_forms(captured) for v in np.flatnonzero(counts)) + (
                7 if any("eri_group_fused" in k for k in captured) else 0) >= np.count_nonzero(counts)
            build(h, run)
            h.destroy()


def scenario_asked_tile_lengths_hold(host):
    """LIBERI_OPT_TILE_LEN: every row-tiled class has tiles of that length, also
    the classes of few quartets, which otherwise run one workgroup step a tile;
    the statistics give the length of either."""
    from gms_liberi_amd import liberi

    b = cluster(17, 5)
    d = np.zeros(b.ntri)
    h = liberi.Handle()
    h.setup(b)
    h.set_option(liberi.OPT_GRAPH, 0)
    longest = {}
    for length in (0, 512, 1024, 4096, 16384, 0):
        h.set_option(liberi.OPT_TILE_LEN, length)
        for lines in (1, 2):
            h.set_option(liberi.OPT_ROW_TILES, 2)  # (no shared launches)
            host.log()
            h.fock_build(d)
        lines = [x for x in host.log() if x.startswith("launch")]
        assert not any("GRID" in x for x in lines)
        forms = launched_forms(lines)
        tile = h.stats()["class_tile"]
        rows = [c for c in forms if forms[c][0] in (1, 2)]
        assert len(rows) >= 12
        assert all(field(x, "quartets") == field(x, "share") for x in lines if "tiles=" in x)
        for c in rows:
            assert forms[c][1] <= tile[c], (length, c)
            assert tile[c] == length if length else tile[c] <= 512, (length, c)
        longest[length] = {c: forms[c][1] for c in rows}
    # rows of up to 647 quartets: whole where the length allows
    assert max(longest[512].values()) == 512 < max(longest[1024].values())
    for c, n in longest[16384].items():
        for length in (512, 1024, 4096):
            assert longest[length][c] == min(n, length), (length, c)
    h.destroy()


def scenario_setup_keeps_to_the_device_budget(host):
    """LIBERI_OPT_MAX_DEVICE_BYTES: no moment of a setup holds more than the
    budget, whether it succeeds or not, and the handle's resident bytes are
    enough of a budget."""
    from gms_liberi_amd import liberi

    for b in (golden("cfg_water.npz"), golden("cfg_ethane.npz"), golden("cfg_cn_chain.npz"), cluster(12, 21)):
        h = liberi.Handle()
        before = host.c.host_bytes()
        h.setup(b)
        full = h.stats()["device_bytes"]
        assert full >= host.c.host_bytes() - before  # all that is held is counted
        quartets = h.stats()["quartets"]
        h.cleanup()
        for budget in [full + x for x in (1 << 20, 1 << 16, 1 << 12, 0, -1, -1000)] + [int(full * x / 40) for x in
                                                                                     range(4, 40)]:
            h.set_option(liberi.OPT_MAX_DEVICE_BYTES, budget)
            before = host.c.host_bytes()
            host.c.host_clear_peak()
            try:
                h.setup(b)
            except liberi.LiberiError as e:
                assert e.code == 5 and budget < full, budget - full
                assert host.c.host_bytes() == before
            else:
                assert budget >= full and np.array_equal(h.stats()["quartets"], quartets)
                h.cleanup()
            assert host.c.host_peak() - before <= budget, (budget - full, host.c.host_peak() - before - budget)
        h.set_option(liberi.OPT_MAX_DEVICE_BYTES, 0)
        h.destroy()


def scenario_statistics_after_a_cleanup(host):
    """A build whose statistics were not read leaves nothing to read once the
    handle's data is gone."""
    from gms_liberi_amd import liberi

    b = golden("cfg_water.npz")
    n = b.ntri
    s = host.stream()
    D, F = host.array(np.zeros(n)), host.array(np.zeros(n))
    for opt, value in ((liberi.OPT_FP32_TAU, 1e-6), (liberi.OPT_CLASS_TIMING, 1)):
        h = liberi.Handle()
        h.setup(b)
        h.set_option(opt, value)
        for end in (h.cleanup, lambda: h.setup(b)):
            if not h.is_initialized:
                h.setup(b)
            h.fock_build_device(D.value, F.value, n, s.value)
            end()
            st = h.stats()
            assert st["last_build_ms"] == 0 and st["fp32_quartets"] == 0 and not st["class_ms"].any()
        h.destroy()


def scenario_footprint_estimate_is_an_upper_bound(host):
    """The bytes that admit a request cover what its handle holds after a build,
    from a few quartets to many for the number of pairs."""
    from gms_liberi_amd import liberi, serving

    for b in (golden("cfg_water.npz"), golden("cfg_ethane.npz"), golden("cfg_cn_chain.npz"), golden("cfg_c60.npz"),
              cluster(17, 5), cluster(30, 6), row_of_s(100), row_of_s(300, 0.02)):
        h = liberi.Handle()
        before = host.c.host_bytes()
        h.setup(b)
        h.fock_build(np.zeros(b.ntri))
        held = host.c.host_bytes() - before
        assert held <= h.stats()["device_bytes"] <= serving.estimate_device_bytes(b), b.num_bas
        h.destroy()


def scenario_outstanding_builds_are_bounded(host):
    """A caller that never waits has at most 16 builds of a handle outstanding,
    and the device at least 8 to go on with after every wait."""
    from gms_liberi_amd import liberi

    b = golden("cfg_water.npz")
    n = b.ntri
    D, F, Da, Db, Fa, Fb = (host.array(np.zeros(n)) for _ in range(6))
    for graph in (1, 0):
        h = liberi.Handle()
        h.setup(b)
        h.set_option(liberi.OPT_GRAPH, graph)
        s = host.stream()
        h.fock_build_device(D.value, F.value, n, s.value)
        first = host.c.host_outstanding(s)
        h.fock_build_device(D.value, F.value, n, s.value)
        per = host.c.host_outstanding(s) - first  # work items of a build
        most, least = 0, 10 ** 9
        for k in range(1, 200):
            h.fock_build_device(D.value, F.value, n, s.value)
            now = host.c.host_outstanding(s)
            most = max(most, now)
            if k > 20:
                least = min(least, now)
        assert most <= 16 * per + first and least >= 8 * per, (graph, most, least, per)
        for _ in range(100):
            assert h._lib.liberi_c_fock_build_uhf_device(h._h, Da, Db, Fa, Fb, n, s) == 0
            assert host.c.host_outstanding(s) <= 16 * (2 * per + 1) + 2 * first
        h.destroy()


SCENARIOS = [k[len("scenario_"):] for k in list(globals()) if k.startswith("scenario_")]


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_host_calls(scenario, host_lib):
    run(scenario, host_lib)


if __name__ == "__main__":
    globals()["scenario_" + sys.argv[2]](Host(sys.argv[1]))
