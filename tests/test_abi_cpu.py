"""Host-side checks of the C ABI that need no GPU: the library loads, exports
every symbol include/ixhip.h declares, and refuses malformed requests before
any kernel launch."""
import ctypes as C
import os
import re

import pytest
import torch

from ixrun_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols(header="ixhip.h"):
    text = open(os.path.join(ROOT, "include", header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ixh_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_exported():
    lib = _lib.lib()
    names = declared_symbols()
    assert "ixh_gemv" in names and "ixh_decode" in names and "ixh_prefix_build" in names
    for name in names:
        assert hasattr(lib, name), f"{name} is declared in include/ixhip.h but not exported"
    assert set(_lib.EXPORTS) == set(names)
    assert lib.ixh_version() >= 100


def test_option_setter_is_not_in_the_product_header():
    """The process-wide kernel-selection switches are a testing hook: the product header declares no setter (nor
    mentions one), the test header declares exactly that one symbol, and the binding reads nothing from the
    environment but the library's path."""
    public = open(os.path.join(ROOT, "include", "ixhip.h")).read()
    assert "set_option" not in public and "option" not in " ".join(declared_symbols())
    assert declared_symbols("ixhip_test.h") == ["ixh_set_option"] == list(_lib.TEST_EXPORTS)
    assert hasattr(_lib.lib(), "ixh_set_option")
    pkg = os.path.join(ROOT, "ixrun_amd")
    reads = []
    for name in sorted(os.listdir(pkg)):
        if name.endswith(".py"):
            text = open(os.path.join(pkg, name)).read()
            reads += [(name, var) for var in re.findall(r"environ(?:\.get)?[\[(]\s*\"([A-Z_0-9]+)\"", text)]
    assert reads == [("_lib.py", "IXH_LIB")], reads


def _packed(level_bits=(3, 5, 8), out_f=4, in_f=8, bm0_words=1):
    s = _lib.IxhPacked()
    s.n_levels = len(level_bits)
    for i, b in enumerate(level_bits):
        s.level_bits[i] = b
    s.out_f, s.in_f = out_f, in_f
    s.bitmaps[0] = 0x1000
    s.bitmap_words[0] = bm0_words
    s.scale = 0x1000
    return s


def test_entries_and_workspace_sizes():
    lib = _lib.lib()
    assert lib.ixh_prefix_entries(10, 5) == 3 and lib.ixh_prefix_entries(11, 5) == 4
    assert lib.ixh_prefix_entries(0, 512) == 1 and lib.ixh_prefix_entries(10, 0) == -1
    s = _packed(out_f=8, in_f=2048, bm0_words=512)
    assert lib.ixh_gemv_workspace_bytes(C.byref(s), 512, 3, 0) == 4 * 3 * 8 * 4
    assert lib.ixh_gemv_workspace_bytes(C.byref(s), 2048, 3, 0) == 0
    assert lib.ixh_gemv_workspace_bytes(C.byref(s), 512, 3, _lib.IXH_GEMV_ATOMIC) == 0


def test_noalloc_entry_rejects_oversize_on_the_host():
    """ixh_gemv_noalloc refuses, before any GPU call, a request whose partial sums exceed its built-in buffer, and
    the atomic mode (which takes no workspace)."""
    lib = _lib.lib()
    s = _packed(out_f=1 << 14, in_f=1 << 14, bm0_words=1 << 23)
    assert lib.ixh_gemv_workspace_bytes(C.byref(s), 512, 16, 0) == 32 * 16 * (1 << 14) * 4 > (16 << 20)
    rc = lib.ixh_gemv_noalloc(C.byref(s), 0x1000, 512, 0x1000, 16, 1 << 14, 0x1000, 1 << 14, 0, None)
    assert rc == -4 and b"built-in buffer" in lib.ixh_last_error()
    rc = lib.ixh_gemv_noalloc(C.byref(s), 0x1000, 512, 0x1000, 1, 1 << 14, 0x1000, 1 << 14, _lib.IXH_GEMV_ATOMIC, None)
    assert rc == -1


@pytest.mark.parametrize("mutate,needle", [
    (lambda s: setattr(s, "n_levels", 1), "n_levels"),
    (lambda s: s.level_bits.__setitem__(2, 7), "last level"),
    (lambda s: s.level_bits.__setitem__(0, 6), "ascend"),
    (lambda s: setattr(s, "out_f", 1 << 20) or setattr(s, "in_f", 1 << 12), "31-bit"),
    (lambda s: s.bitmap_words.__setitem__(0, 0), "bitmap 0"),
    (lambda s: setattr(s, "scale", None), "scale"),
])
def test_malformed_packed_is_refused(mutate, needle):
    lib = _lib.lib()
    s = _packed()
    mutate(s)
    rc = lib.ixh_decode(C.byref(s), 0x1000, 8, None, 0x1000, None)
    assert rc == -1 and needle in lib.ixh_last_error().decode()


@pytest.mark.parametrize("change,group,out,needle", [
    ({}, 64, 0x1000, None),
    ({}, None, 0x1000, None),
    ({"level_bits": (3, 4, 5, 6, 8)}, None, 0x1000, "(3,5,8)"),
    ({"in_f": (1 << 11) + 1}, None, 0x1000, "2^22"),
    ({"out_f": 1, "in_f": (1 << 22) + 1}, None, 0x1000, "2^22"),
    ({"last": 0x1002}, None, 0x1000, "last stream"),
    ({}, None, 0x1008, "16-byte"),
    ({}, 16, 0x1000, "power of two"),
    ({}, 96, 0x1000, "power of two"),
    ({"named": 3}, None, 0x1000, "named"),
])
def test_decode_without_a_table_says_what_it_does_not_take(change, group, out, needle):
    """Each call that is refused is refused with its own reason, before any launch; asking first leaves the last error as it was."""
    lib = _lib.lib()
    change = dict(change)
    named, last = change.pop("named", 0), change.pop("last", 0x1000)
    s = _packed(**{"out_f": 1 << 11, "in_f": 1 << 11, "bm0_words": (1 << 17) + 64, **change})
    s.last, s.last_bytes = last, 4
    scales = 0x1000 if group else None
    assert lib.ixh_set_option(b"decode_kernel", named) == 0
    try:
        assert lib.ixh_decode_unranked(None, None, 0, 0x1000, None) == -1
        before = lib.ixh_last_error()
        assert lib.ixh_decode_unranked_takes(C.byref(s), scales, group or 0, out) == (needle is None)
        assert lib.ixh_last_error() == before
        if needle:
            assert lib.ixh_decode_unranked(C.byref(s), scales, group or 0, out, None) == -2
            assert needle in lib.ixh_last_error().decode()
    finally:
        lib.ixh_set_option(b"decode_kernel", 0)


def test_malformed_gemv_arguments():
    lib = _lib.lib()
    s = _packed(out_f=4, in_f=1024, bm0_words=128)
    call = lambda chunk, m, x=0x1000, y=0x1000, ws=None, wsb=0, flags=0: lib.ixh_gemv(
        C.byref(s), 0x1000, chunk, x, m, 1024, y, 4, None, ws, wsb, flags, None)
    assert call(512, 0) == -1 and "m = 0" in lib.ixh_last_error().decode()
    assert call(512, 17) == -1
    assert call(500, 1) == -1 and "divide" in lib.ixh_last_error().decode()
    assert call(512, 1, x=None) == -1
    assert call(512, 1, y=None) == -1
    assert call(512, 1) == -4 and "workspace" in lib.ixh_last_error().decode()  # two chunks need partial sums
    assert call(512, 1, flags=_lib.IXH_GEMV_ATOMIC) == -1 and "y32" in lib.ixh_last_error().decode()
    with pytest.raises(_lib.IxhError):
        _lib.check(-1)


def test_malformed_encode_arguments():
    lib = _lib.lib()
    bits = (C.c_int32 * 3)(3, 5, 8)
    need = lib.ixh_encode_workspace_bytes(4, 1024, 3)
    assert need >= 1024 + 2 * 4  # 256 partial maxima and one tile sum for each of the two table rows
    assert lib.ixh_encode_workspace_bytes(0, 1024, 3) == 0 and lib.ixh_encode_workspace_bytes(4, 1024, 9) == 0
    scan = lambda out_f=4, in_f=1024, nl=3, lb=bits, w=0x1000, sc=0x1000, tab=0x1000, ws=0x1000, wsb=need: \
        lib.ixh_encode_scan(w, out_f, in_f, nl, lb, sc, tab, ws, wsb, None)
    assert scan(nl=1) == -1 and "n_levels" in lib.ixh_last_error().decode()
    assert scan(lb=(C.c_int32 * 3)(3, 5, 7)) == -1 and "last level" in lib.ixh_last_error().decode()
    assert scan(lb=(C.c_int32 * 3)(5, 3, 8)) == -1 and "ascend" in lib.ixh_last_error().decode()
    assert scan(out_f=0) == -1 and "empty" in lib.ixh_last_error().decode()
    assert scan(out_f=1 << 20, in_f=1 << 12) == -1 and "31-bit" in lib.ixh_last_error().decode()
    assert scan(w=None) == -1 and scan(sc=None) == -1 and scan(tab=None) == -1
    assert scan(wsb=need - 1) == -4 and "workspace" in lib.ixh_last_error().decode()
    s = _packed(out_f=4, in_f=1024, bm0_words=128)
    assert lib.ixh_encode_pack(None, C.byref(s), 0x1000, None) == -1
    assert lib.ixh_encode_pack(0x1000, C.byref(s), None, None) == -1
    s.bitmap_words[0] = 3
    assert lib.ixh_encode_pack(0x1000, C.byref(s), 0x1000, None) == -1 and "bitmap 0" in lib.ixh_last_error().decode()


def test_device_packed_refuses_cpu_tensors():
    from ixrun_amd.quantize import int8x_quantize

    p = int8x_quantize((torch.randn(8, 64) * 0.02).bfloat16())
    with pytest.raises(RuntimeError, match="GPU"):
        _lib.DevicePacked(p["level_bits"], 8, 64, p["bitmaps"], p["streams"], p["scale"].reshape(1))


def test_missing_library_is_loud(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", "/nonexistent/libixhip.so")
    with pytest.raises(RuntimeError, match="no fallback"):
        _lib.lib()


def load_bench():
    import sys

    sys.path.insert(0, ROOT)
    try:
        import bench
    finally:
        sys.path.remove(ROOT)
    return bench


def test_bench_counts_the_form_that_is_read():
    """bench.py divides the bytes of what a forward reads: the lane layout where the rows go there (its listed elements, not
    the list's spare room), the packed streams otherwise."""
    from types import SimpleNamespace as Of

    bench = load_bench()
    packed = {"total_bytes": 44}
    off = torch.tensor([0, 3, 7], dtype=torch.int32)
    lanes = Of(tensors=(torch.zeros(640, dtype=torch.int32), off, torch.zeros(400, dtype=torch.int16), torch.zeros(400, dtype=torch.int8)))
    layer = Of(_lanes=lanes, _gemm_ok=True, _fused_plan=lambda rows: (rows < 8, ((0, rows, 0),), False) if rows <= 16 else False,
               _lanes_gemm_wins=lambda rows: rows < 100)
    read = 640 * 4 + 3 * 4 + 7 * 12
    assert [bench.form_read(layer, packed, m) for m in (1, 50)] == [("lanes", read)] * 2
    assert [bench.form_read(layer, packed, m) for m in (8, 200)] == [("packed", 44)] * 2
    layer._gemm_ok = False
    assert bench.form_read(layer, packed, 50) == ("packed", 44)
    layer._lanes = None
    assert bench.form_read(layer, packed, 50) == ("packed", 44)


def test_bench_tables_are_well_formed():
    """bench.py's workload table (shape, rows, recipe[, level scheme]) and its table of measured HBM traffic, whose
    entries name sources that exist and workloads that the first table holds."""
    bench, root = load_bench(), ROOT
    for name, spec in bench.WORKLOADS.items():
        assert len(spec) in (4, 5), name
        out_f, in_f, m, recipe = spec[:4]
        assert isinstance(out_f, int) and isinstance(in_f, int) and isinstance(m, int) and isinstance(recipe, str), name
        assert out_f > 0 and in_f > 0 and 0 <= m <= 512, name  # m = 0: decode and encode workloads
    for name, (nbytes, files, sha16) in bench.MEASURED_TRAFFIC_BYTES.items():
        assert nbytes > 0 and isinstance(sha16, str), name
        assert name.removesuffix("_unfused").removesuffix("_packed") in bench.WORKLOADS, name
        for f in files:
            assert os.path.exists(os.path.join(root, "ixrun_amd", "csrc", f)), (name, f)


def test_bench_counter_runs_are_of_the_form_that_is_read():
    """A product's counters are those of the lanes' kernels under its own name, and of the kernels that read the packed streams
    under a name of theirs, whatever the number of rows."""
    bench = load_bench()
    assert [bench.counted_as("w", form) for form in ("lanes", "packed")] == ["w", "w_packed"]
    assert bench.counted_as("w", "packed", unfused=True) == "w_unfused"
    for table in (bench.MEASURED_TRAFFIC_BYTES, bench.MEASURED_INSTRUCTIONS):
        for name, (_, files, _) in table.items():
            base = name.removesuffix("_unfused").removesuffix("_packed")
            if bench.WORKLOADS[base][2] and files:  # (0 rows: decode and encode)
                assert (name == base) == any("lanes" in f for f in files), name


def test_malformed_lane_layouts():
    """Descriptors that a kernel could not read within its buffers are refused on the host: the list is whole groups of 64
    quads, at least one."""
    lib = _lib.lib()
    words = lib.ixh_lanes_plane_words(8, 1024, 3)
    assert words == 2 * 2 * 64 * 3 and lib.ixh_lanes_cells(8, 1024) == 4
    good = lambda: _lib.IxhLanes(3, 8, 1024, 0x1000, words, 0x1000, 0x1000, 0x1000, 64, 0x1000)
    assert lib.ixh_lanes_gemv_workspace_bytes(C.byref(good()), 16) >= 0
    call = lambda s: lib.ixh_lanes_gemv(C.byref(s), 0x1000, 1024, None, 1, 0x1000, 8, None, 0, None)
    for field, value, needle in (("n_quads", 0, "groups of 64"), ("n_quads", 63, "groups of 64"), ("n_quads", 65, "groups of 64"),
                                 ("n_quads", 1 << 30, "2^30"), ("exc_pos", None, "NULL"), ("plane_words", words - 1, "plane"),
                                 ("plane", 0x1004, "16-byte"), ("bits", 6, "no lane layout"), ("in_f", 1 << 31, "no lane layout")):
        s = good()
        setattr(s, field, value)
        assert call(s) == -1 and needle in lib.ixh_last_error().decode(), (field, value, lib.ixh_last_error())


def test_several_rows_of_many_row_quads_are_not_the_gemv_kernels():
    """Three and four rows of layers of more than 30 row quads a CU go to the kernel of 16 weight rows a wave (told by the scratch that it
    takes on a layer of this size, where the one-row kernel takes none)."""
    lib = _lib.lib()

    def need(out_f, in_f, bits, rows):
        words = lib.ixh_lanes_plane_words(out_f, in_f, bits)
        s = _lib.IxhLanes(bits, out_f, in_f, 0x1000, words, 0x1000, 0x1000, 0x1000, 64, 0x1000)
        return lib.ixh_lanes_gemv_workspace_bytes(C.byref(s), rows)

    assert need(65536, 5120, 5, 3) > 0 and need(65536, 5120, 5, 4) > 0
    assert need(65536, 5120, 5, 1) == 0 and need(17408, 5120, 5, 4) == 0
