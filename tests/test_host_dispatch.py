"""Host side of the launches on a machine without a GPU: which kernel a call
takes, what it allocates and what it refuses.

The library is loaded over a stand-in for the HIP runtime (fake_hip.cpp),
which records launches instead of running them, in a process of its own: the
file runs itself with the case's name.  256 CUs of 160 KB LDS, 16 resident
one-wave workgroups a CU."""
from __future__ import annotations

import ctypes as C
import importlib.util
import os
import re
import shutil
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
LIB = ROOT / "go-fann_amd" / "libgofann_hip.so"

GIB = 1 << 30
SIDE = 0x1000  # a stream that is not the default one


class Fake:
    """The library over the stand-in runtime."""

    def __init__(self, stub: str):
        self.hip = C.CDLL(stub, mode=os.RTLD_NOW | os.RTLD_GLOBAL)
        self.hip.fake_limit.argtypes = [C.c_size_t]
        self.hip.fake_used.restype = C.c_size_t
        self.hip.fake_name.restype = C.c_char_p
        self.hip.fake_capture.argtypes = [C.c_void_p]
        spec = importlib.util.spec_from_file_location(
            "_lib", ROOT / "go-fann_amd" / "gofann_amd" / "_lib.py")
        self.L = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(self.L)
        self.lib = self.L.load()
        self.mem = C.create_string_buffer(1 << 20)  # what every "device array" points to
        self.p = (C.addressof(self.mem) + 255) & ~255

    def context(self, stream=0):
        h = self.L.P()
        assert self.lib.gofann_create(0, C.byref(h)) == 0
        assert self.lib.gofann_set_stream(h, self.L.P(stream)) == 0
        return h

    def launched(self):
        """Names and grids of the launches since the last call."""
        out = [(self.hip.fake_name(i).decode(), self.hip.fake_grid(i))
               for i in range(self.hip.fake_launches())]
        self.hip.fake_clear()
        return out

    group_rows = 100_000  # rows a group of the graphs

    def graph(self, degree=32):
        L, p = self.L, self.p
        return L.GraphView(p, p, p, 3 * self.group_rows, degree, 3, 1000, None)

    def routes(self, count):
        p = self.p
        return self.L.Routes(p, p, p, None, None, None, None, None, None, 0, count, None)

    def exact(self, ctx, elem, dim, beam, count, place=0):
        L, p = self.L, self.p
        return self.lib.gofann_exact_search(ctx, p, elem, dim, 1000, p, self.graph(), None,
                                            L.PredicateView(), self.routes(count),
                                            L.ExactParams(beam, 1, 2, 0, 10, place), p, p, None)

    def exact_scan(self, ctx, routes):
        p = self.p
        return self.lib.gofann_exact_posting_scan(
            ctx, p, self.L.ELEM_F32, 64, 1000, p, self.L.PredicateView(), p, p, p, p, routes, 10,
            self.L.EXACT_ORDER_SERIAL, p, p, None)

    def rabitq(self, ctx, bits, beam, count):
        L, p = self.L, self.p
        rq = L.RabitqView(p, p, p, p, bits, bits, 64, 1000, None, 0)
        prm = L.SearchParams(beam, 1, 2, 0, 10, 100, 0.0, 0.0, 0, 0, 0, 0)
        return self.lib.gofann_rabitq_search(ctx, rq, L.RabitqQueries(p, p, p, p, p, 16),
                                             self.graph(), L.PredicateView(), self.routes(count),
                                             prm, p, p, None)

    def pq(self, ctx, m, beam, count):
        L, p = self.L, self.p
        prm = L.SearchParams(beam, 1, 2, 0, 10, 100, 0.0, 0.0, 0, 0, 0, 0)
        return self.lib.gofann_pq_search(ctx, L.PqView(p, p, 4 * m, m, 1000, None, 0), p,
                                         L.ELEM_F32, self.graph(), L.PredicateView(),
                                         self.routes(count), prm, p, p, None)

    def placement(self, ctx):
        """(PQ table in LDS, visited placement) of the last launch."""
        v = [C.c_int() for _ in range(4)]
        assert self.lib.gofann_last_placement(ctx, *[C.byref(x) for x in v]) == 0
        return v[0].value, ("global", "lds", "spill")[v[1].value]


def exact_kernel(name: str):
    """(visited placement, set registers) of an exact-route kernel's name."""
    m = re.search(r"exact_(route|set)_kernelILi(\d)ELin?\d+ELi\d+E(?:Li(\d)E)?E", name)
    assert m, name
    return {0: "global", 1: "lds", 2: "spill"}[int(m.group(2))], int(m.group(3) or 0)


# --------------------------------------------------------------------------
# Cases (run in the child process)
# --------------------------------------------------------------------------
def case_rings_without_slabs(f: Fake):
    """20,000 f32 routes whose rings fit in memory and whose visited slabs
    then do not: the heap frontier takes them, and the rings are given back."""
    ctx = f.context()
    slabs, rings = 20_000 * 16384, 20_000 * 2048 * 8
    f.hip.fake_limit(f.hip.fake_used() + rings + slabs // 2)
    assert f.exact(ctx, f.L.ELEM_F32, 64, 300, 20_000) == f.L.OK
    [(name, grid)] = f.launched()
    assert exact_kernel(name)[1] == 0 and grid == 20_000
    assert f.hip.fake_used() <= slabs + 1024
    # with room for both, the set frontier
    f.hip.fake_limit(8 * GIB)
    assert f.exact(ctx, f.L.ELEM_F32, 64, 300, 20_000) == f.L.OK
    [(name, _)] = f.launched()
    assert exact_kernel(name)[1] == 8


def case_rings_are_bounded(f: Fake):
    """A launch whose rings would pass 2 GiB takes the heap frontier."""
    ctx = f.context()
    for count, regs in ((1 << 17, 8), ((1 << 17) + 1, 0)):
        assert f.exact(ctx, f.L.ELEM_F16, 64, 300, count) == f.L.OK
        [(name, _)] = f.launched()
        assert exact_kernel(name)[1] == regs


def case_capture_elsewhere(f: Fake):
    """A search or a scan that allocates its optional buffers while another
    stream is captured leaves that capture intact."""
    for call in (lambda h: f.exact(h, f.L.ELEM_F32, 64, 96, 8, f.L.PLACE_LDS),
                 lambda h: f.exact_scan(h, 8)):
        f.hip.fake_capture(0x2000)
        assert call(f.context(SIDE)) == f.L.OK
        assert not f.hip.fake_capture_broken()
        f.hip.fake_capture(None)


def case_captured_launches_keep_no_scratch(f: Fake):
    """Under capture neither allocates: the heap frontier, and one workgroup
    a route."""
    f.hip.fake_capture(SIDE)
    h, used = f.context(SIDE), f.hip.fake_used()
    assert f.exact(h, f.L.ELEM_F32, 64, 96, 8, f.L.PLACE_LDS) == f.L.OK
    [(name, _)] = f.launched()
    assert exact_kernel(name) == ("lds", 0)
    assert f.exact_scan(h, 8) == f.L.OK
    [(name, grid)] = f.launched()
    assert "exact_scan_kernel" in name and grid == 8
    assert f.hip.fake_used() == used and not f.hip.fake_capture_broken()
    f.hip.fake_capture(None)
    # outside it: 16 runs a route and their merge
    assert f.exact_scan(h, 8) == f.L.OK
    assert [g for _, g in f.launched()] == [128, 8]


def case_bucket_reps_without_memory(f: Fake):
    """Bucket representatives need no buffer: without memory for the keys, one
    workgroup per bucket."""
    h = f.context()
    off = (C.c_uint32 * 5)(0, 8, 16, 24, 32)
    for limit, kernels in ((0, ["bucket_rep_kernel"]),
                           (GIB, ["bucket_mean_kernel", "bucket_dist_kernel",
                                  "bucket_pick_kernel"])):
        f.hip.fake_limit(f.hip.fake_used() + limit)
        assert f.lib.gofann_build_bucket_reps(h, f.p, f.L.ELEM_F32, 64, C.addressof(off), 4, f.p,
                                              f.p) == f.L.OK
        names = [n for n, _ in f.launched()]
        assert len(names) == len(kernels) and all(k in n for k, n in zip(kernels, names)), names


def case_u8_set_frontier(f: Fake):
    """u8 rows take the set frontier up to 16 routes and Q = 112, float rows at
    any number and up to Q = 496."""
    h = f.context()
    for elem, beam, count, regs in ((f.L.ELEM_U8, 112, 16, 2), (f.L.ELEM_U8, 113, 1, 0),
                                    (f.L.ELEM_U8, 2, 17, 0), (f.L.ELEM_U8, 200, 16, 0),
                                    (f.L.ELEM_F16, 112, 999, 2), (f.L.ELEM_F16, 113, 1, 4),
                                    (f.L.ELEM_F32, 240, 17, 4), (f.L.ELEM_F32, 241, 17, 8),
                                    (f.L.ELEM_F32, 496, 1, 8), (f.L.ELEM_F32, 497, 1, 0)):
        assert f.exact(h, elem, 64, beam, count) == f.L.OK
        [(name, _)] = f.launched()
        assert exact_kernel(name)[1] == regs, (elem, beam, count)


def case_full_table_beside_others(f: Fake):
    """The full LDS table: every resident launch on the default stream; up to
    a quarter of a CU's LDS on a stream that may run beside others."""
    for stream, per_cu, want in ((0, 1, "lds"), (0, 5, "lds"), (SIDE, 1, "lds"),
                                 (SIDE, 2, "lds"), (SIDE, 3, "spill"), (SIDE, 5, "spill")):
        h = f.context(stream)
        assert f.exact(h, f.L.ELEM_F32, 64, 64, per_cu * 256) == f.L.OK
        assert f.placement(h)[1] == want, (stream, per_cu)
        assert f.rabitq(h, 512, 64, per_cu * 256) == f.L.OK
        assert f.placement(h)[1] == want, (stream, per_cu)
        # 28 KB a route (4096 bits, Q = 320): one a CU
        assert f.rabitq(h, 4096, 320, per_cu * 256) == f.L.OK
        want = "lds" if stream == 0 or per_cu == 1 else "global"
        assert f.placement(h)[1] == want, (stream, per_cu)


def case_pq_form(f: Fake):
    """PQ's form (table in LDS or entries on demand) does not depend on the
    visited placement that a launch of the size takes: with 16 subspaces the
    entries on demand hold twice the routes of the table (16 a CU, 8), also
    where their full table holds only 8."""
    for count in (1, 1000, 1800, 2048, 2049, 9000):
        h = f.context()
        assert f.pq(h, 16, 64, count) == f.L.OK
        assert f.placement(h) == (0, "lds" if count <= 2048 else "spill"), count


def case_narrow_beams_spill(f: Fake):
    """A narrow beam's launch that the spilling table holds (21 routes a CU)
    takes it, though the slab would hold more (28)."""
    f.hip.fake_waves(28)
    h = f.context()
    for rows, beam, count, want in ((8193, 80, 21 * 256, "spill"), (8193, 81, 21 * 256, "global"),
                                    (8192, 81, 21 * 256, "spill"), (8192, 129, 5000, "global"),
                                    (8192, 80, 21 * 256 + 1, "global")):
        f.group_rows = rows
        assert f.pq(h, 32, beam, count) == f.L.OK
        assert f.placement(h)[1] == want, (rows, beam, count)
    # exact f32 rows, dim 3072: 8 or 9 a CU against 10 or more; full table: 4
    for rows, beam, want in ((8192, 224, "spill"), (8192, 225, "global"), (8193, 160, "spill"),
                             (8193, 161, "global")):
        f.group_rows = rows
        assert f.exact(h, f.L.ELEM_F32, 3072, beam, 1500) == f.L.OK
        assert f.placement(h)[1] == want, (rows, beam)


def case_most_residents(f: Fake):
    """Past the full table, the most resident routes a CU, also where the
    spilling table holds the whole launch."""
    h = f.context()
    assert f.rabitq(h, 512, 384, 2584) == f.L.OK      # spill 13 a CU, slab 16
    assert f.placement(h)[1] == "global"
    assert f.exact(h, f.L.ELEM_F16, 512, 416, 2584) == f.L.OK
    assert f.placement(h)[1] == "global"
    # 16 KB rows: 6 with the spilling table, 7 with the slab
    assert f.exact(h, f.L.ELEM_F32, 4096, 352, 3333) == f.L.OK
    assert f.placement(h)[1] == "global"


def case_lds_granules(f: Fake):
    """LDS comes in granules of 1280 bytes: 32,396 a route (f32, dim 3072, Q =
    256, full table) are 26 of 128, four routes a CU and not the five that
    the bytes allow."""
    h = f.context()
    assert f.exact(h, f.L.ELEM_F32, 3072, 256, 4 * 256) == f.L.OK
    assert f.placement(h)[1] == "lds"
    assert f.exact(h, f.L.ELEM_F32, 3072, 256, 4 * 256 + 1) == f.L.OK
    assert f.placement(h)[1] != "lds"


def case_u8_slabs(f: Fake):
    """u8 rows, 25 a CU with the spilling table and 28 with the slab: the
    spilling table at Q <= 64, past a round of residents at Q <= 72, past two
    where a step reads 8 KB of rows."""
    f.hip.fake_waves(28)
    h, round_ = f.context(), 28 * 256

    def placed(dim, degree, beam, count):
        L, p = f.L, f.p
        assert f.lib.gofann_exact_search(
            h, p, L.ELEM_U8, dim, 1000, p, f.graph(degree), None, L.PredicateView(),
            f.routes(count), L.ExactParams(beam, 1, 2, 0, 10, 0), p, p, None) == L.OK
        return f.placement(h)[1]
    # narrow beams by the rows a group
    for rows, beam, want in ((8192, 160, "spill"), (8192, 161, "global"), (16384, 112, "spill"),
                             (16384, 113, "global"), (16385, 64, "spill"), (16385, 65, "global")):
        f.group_rows = rows
        assert placed(192, 32, beam, 4000) == want, (rows, beam)
    f.group_rows = 100_000
    # (the rows' LDS pads the spilling table to 25 a CU)
    for dim, degree, beam, count, want in (
            (1088, 4, 64, 5000, "spill"), (1088, 8, 65, 5000, "global"),
            (1088, 8, 72, round_, "global"), (1088, 8, 72, round_ + 1, "spill"),
            (1088, 8, 73, 2 * round_, "global"), (1088, 8, 73, 2 * round_ + 1, "spill"),
            (1088, 6, 73, 2 * round_ + 1, "global"), (1088, 6, 72, round_ + 1, "spill"),
            (1088, 8, 100, 2 * round_ + 1, "spill"),    # 21 a CU: a third of it more
            (1088, 8, 160, 2 * round_ + 1, "global"),   # 18 a CU
            (192, 64, 300, 60_000, "global")):
        assert placed(dim, degree, beam, count) == want, (dim, degree, beam, count)


# --------------------------------------------------------------------------
CASES = sorted(k[5:] for k in globals() if k.startswith("case_"))


def pytest_generate_tests(metafunc):
    if "case" in metafunc.fixturenames:
        metafunc.parametrize("case", CASES)


def _stub(tmp: Path) -> Path:
    out = tmp / "libfake_hip.so"
    if not out.exists():
        cxx = shutil.which("g++") or "g++"
        subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", str(ROOT / "tests" / "fake_hip.cpp"),
                        "-o", str(out)], check=True, timeout=300)
    return out


def test_dispatch(case, hip_lib_path, tmp_path_factory):
    base = tmp_path_factory.getbasetemp() / "fake_hip"
    base.mkdir(exist_ok=True)
    res = subprocess.run([sys.executable, __file__, case, str(_stub(base))], timeout=120,
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stdout[-2000:] + res.stderr[-2000:]


if __name__ == "__main__":
    globals()["case_" + sys.argv[1]](Fake(sys.argv[2]))
