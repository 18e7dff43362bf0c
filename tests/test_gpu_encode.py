"""The device encoder against the CPU oracle and the CPU writer, through the C ABI.

Everything here is integer / byte work and must be bit-exact: the bf16 scale, the
per-level counts, every word of every bitmap and code stream, the last level's bytes and
the rank table at unit 512 (reference: ixrun/quantize.py:41-122, ixrun/bitpack.py:13-61,
ixrun/fused.py:67-78).
"""
import numpy as np
import pytest
import torch

from helpers import bf16_bits, calibrated_weight, outlier_weight, student_t_weight

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from ixrun_amd import _lib

    assert _lib.lib().ixh_version() >= 100
    return torch.device("cuda:0")


def make_weight(kind, out_f, in_f):
    g = torch.Generator("cpu").manual_seed(5)
    if kind == "student_t":
        return student_t_weight(out_f, in_f, seed=0)
    if kind == "outlier":
        return outlier_weight(out_f, in_f, seed=0)
    if kind == "calibrated_pow2":
        return calibrated_weight(out_f, in_f, seed=0)[0]
    if kind == "calibrated_odd_scale":
        return calibrated_weight(out_f, in_f, seed=0, scale=0.0123046875)[0]
    if kind == "zeros":  # the scale falls back to its floor, every value is 0
        return torch.zeros(out_f, in_f, dtype=torch.bfloat16)
    if kind == "all_extreme":  # every element +-max: only the last level is used
        sign = torch.randint(0, 2, (out_f, in_f), generator=g) * 2 - 1
        return (sign * 0.75).bfloat16()
    if kind == "wide_range":  # magnitudes over many binades: quotients near every rounding boundary
        e = torch.randint(-20, 1, (out_f, in_f), generator=g).float()
        return (torch.randn(out_f, in_f, generator=g) * torch.exp2(e)).bfloat16()
    if kind == "tiny":  # near the scale's floor, quotients with subnormal divisors' neighbours
        return (torch.randn(out_f, in_f, generator=g) * 3e-8).bfloat16()
    if kind == "half_steps":  # exact ties k + 0.5 of the quotient: round-half-even decides
        k = torch.randint(-253, 254, (out_f, in_f), generator=g).float() * 0.5
        w = (k * 2.0 ** -7).bfloat16()
        w.view(-1)[0] = 127 * 2.0 ** -7
        return w
    raise KeyError(kind)


KINDS = ["student_t", "outlier", "calibrated_pow2", "calibrated_odd_scale", "zeros", "all_extreme", "wide_range", "tiny",
         "half_steps"]


def oracle_encode(oracle, w, level_bits):
    scale_bits, q = oracle.quantize_bf16(bf16_bits(w))
    e = oracle.encode(q, level_bits)
    table = oracle.prefix(q.size, len(level_bits), e["bitmaps"], 512)
    return scale_bits, q, e, table


def check_against_oracle(oracle, dev, w, level_bits):
    from ixrun_amd.quantize import int8x_quantize_device

    scale_bits, q, e, table = oracle_encode(oracle, w, level_bits)
    p = int8x_quantize_device(w.to(dev), level_bits)
    torch.cuda.synchronize()
    what = f"{tuple(w.shape)} {level_bits}"
    assert int(bf16_bits(p["scale"].reshape(1))[0]) == scale_bits, f"{what}: scale"
    assert p["counts"] == [int(c) for c in e["counts"]], f"{what}: counts"
    assert p["total_bytes"] == e["total_bytes"], f"{what}: total_bytes"
    for i in range(len(level_bits) - 1):
        got_bm = p["bitmaps"][i].cpu().numpy().view(np.uint32)
        got_st = p["streams"][i].cpu().numpy().view(np.uint32)
        assert got_bm.shape == e["bitmaps"][i].shape and np.array_equal(got_bm, e["bitmaps"][i]), f"{what}: bitmap {i}"
        assert got_st.shape == e["streams"][i].shape and np.array_equal(got_st, e["streams"][i]), f"{what}: stream {i}"
    assert np.array_equal(p["streams"][-1].cpu().numpy(), e["last"]), f"{what}: last level"
    assert np.array_equal(p["table512"].cpu().numpy(), table), f"{what}: rank table"
    return p, q


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(1, 1), (2, 5), (3, 11), (7, 33), (1, 512), (1, 513), (33, 1000), (128, 256),
                                   (300, 1031), (64, 1536), (256, 4608)])
def test_encode_bit_exact(oracle, dev, kind, shape):
    check_against_oracle(oracle, dev, make_weight(kind, *shape), (3, 5, 8))


@pytest.mark.parametrize("level_bits", [(3, 4, 5, 6, 8), (2, 8), (4, 8), (7, 8), (1, 2, 3, 4, 5, 6, 7, 8), (3, 3, 8),
                                        (1, 7, 8)])
@pytest.mark.parametrize("kind", ["student_t", "calibrated_odd_scale", "wide_range"])
def test_encode_other_level_schemes(oracle, dev, kind, level_bits):
    check_against_oracle(oracle, dev, make_weight(kind, 300, 1031), level_bits)


def test_encode_hand_known_answer(dev):
    """The 2x5 tensor worked out by hand from the reference's code: v = [0,1,-3,4,-15 | 16,127,-127,3,5], s = 2^-7."""
    from ixrun_amd.quantize import int8x_quantize_device

    v = torch.tensor([0, 1, -3, 4, -15, 16, 127, -127, 3, 5], dtype=torch.float32)
    w = (v * 2.0 ** -7).bfloat16().view(2, 5)
    p = int8x_quantize_device(w.to(dev), (3, 5, 8))
    u32 = lambda t: [int(x) for x in t.cpu().numpy().view(np.uint32)]
    assert u32(p["bitmaps"][0]) == [0x00000107] and u32(p["bitmaps"][1]) == [0x00000023]
    assert u32(p["streams"][0]) == [0x00000C23] and u32(p["streams"][1]) == [0x00005013]
    assert p["streams"][2].cpu().tolist() == [143, 254, 0]
    assert p["counts"] == [4, 3, 3] and p["total_bytes"] == 21
    assert float(p["scale"]) == 2.0 ** -7


def test_encode_matches_cpu_writer(dev):
    """Same dictionary as the package's CPU writer (which follows the reference's writer line by line)."""
    from ixrun_amd.quantize import int8x_quantize, int8x_quantize_device

    w = outlier_weight(96, 1000, seed=3)
    for level_bits in [(3, 5, 8), (3, 4, 5, 6, 8)]:
        a = int8x_quantize(w, level_bits)
        b = int8x_quantize_device(w.to(dev), level_bits)
        for key in ("level_bits", "out_f", "in_f", "N", "counts", "total_bytes", "bits_per_weight", "compression_vs_bf16"):
            assert a[key] == b[key], key
        assert torch.equal(a["scale"], b["scale"].cpu())
        for x, y in zip(a["bitmaps"] + a["streams"], b["bitmaps"] + b["streams"]):
            assert x.dtype == y.dtype and torch.equal(x, y.cpu())


def test_encode_unaligned_weight(oracle, dev):
    """A weight that starts 2 bytes past a 16-byte boundary takes the scalar load path."""
    from ixrun_amd import _lib

    w = student_t_weight(40, 520, seed=2)
    scale_bits, q, e, table = oracle_encode(oracle, w, (3, 5, 8))
    buf = torch.empty(w.numel() + 8, dtype=torch.bfloat16, device=dev)
    view = buf[1 : 1 + w.numel()].view(40, 520)
    view.copy_(w)
    assert view.data_ptr() % 16 == 2
    dp, tab, counts = _lib.encode_device(view, (3, 5, 8))
    assert counts == [int(c) for c in e["counts"]]
    assert np.array_equal(dp.tensors[0].cpu().numpy().view(np.uint32), e["bitmaps"][0])
    assert np.array_equal(dp.tensors[2].cpu().numpy().view(np.uint32), e["streams"][0])
    assert np.array_equal(tab.cpu().numpy(), table)


def test_encode_rejects_bad_arguments(dev):
    from ixrun_amd import _lib
    from ixrun_amd.quantize import int8x_quantize_device

    w = torch.zeros(4, 8, dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError):
        int8x_quantize_device(w, (3, 5, 7))
    with pytest.raises(RuntimeError):
        int8x_quantize_device(w.cpu(), (3, 5, 8))
    with pytest.raises(RuntimeError):
        int8x_quantize_device(torch.zeros(0, 8, dtype=torch.bfloat16, device=dev), (3, 5, 8))
    with pytest.raises(_lib.IxhError):
        _lib.encode_device(w, (3, 9, 8))


@pytest.mark.parametrize("lanes", [True, False])
def test_encoded_layer_runs(oracle, dev, lanes):
    """Encoder output straight into the module: decode gives back the int8, the fused product matches."""
    from ixrun_amd.engine import StreamingLinear
    from ixrun_amd.quantize import int8x_quantize_device

    w = student_t_weight(192, 2048, seed=4)
    p, q = check_against_oracle(oracle, dev, w, (3, 5, 8))
    layer = StreamingLinear(p, lanes=lanes)
    q_dev = torch.empty(p["N"], dtype=torch.int8, device=dev)
    layer._dp.decode(layer._table, layer._unit, out_i8=q_dev)
    assert np.array_equal(q_dev.cpu().numpy(), q)
    x = torch.randn(1, 2048, generator=torch.Generator("cpu").manual_seed(1)).bfloat16()
    y = layer(x.to(dev))
    w_deq = (torch.from_numpy(q.astype(np.float32)) * p["scale"].float().cpu()).bfloat16().view(192, 2048)
    want = torch.nn.functional.linear(x.float(), w_deq.float())
    assert (y.float().cpu() - want).norm() / want.norm() < 4e-3


def test_encode_full_size_layer(oracle, dev):
    """5120x17408 Student-t: every stream equal to the oracle's, and the round trip through the device decoder."""
    from ixrun_amd.triton_kernels import decode_int8

    w = student_t_weight(5120, 17408, seed=0)
    p, q = check_against_oracle(oracle, dev, w, (3, 5, 8))
    assert np.array_equal(decode_int8(p, device=dev).cpu().numpy().reshape(-1), q)


@pytest.mark.parametrize("level_bits", [(3, 5, 8), (1, 8), (3, 4, 5, 6, 8), (1, 2, 3, 4, 5, 6, 7, 8)])
@pytest.mark.parametrize("n", [2016, 2047, 2048, 2049, 2080, 8191, 8192, 8193, 12 * 2048 + 31])
@pytest.mark.parametrize("kind", ["student_t", "half_steps", "zeros", "all_extreme"])
def test_encode_span_edges(oracle, dev, n, level_bits, kind):
    """Around the 2048 elements of a wave and the 8192 of a workgroup, runs that are full, empty or split anywhere."""
    check_against_oracle(oracle, dev, make_weight(kind, 1, n), level_bits)


@pytest.mark.parametrize("level_bits,waves", [((3, 5, 8), 20), ((3, 4, 5, 6, 8), 16), ((2, 8), 24)])
@pytest.mark.parametrize("spans,more", [(1, 0), (1, 1), (2, -1999)])
def test_encode_waves_of_more_than_a_span(oracle, dev, level_bits, waves, spans, more):
    """As many spans of 2048 as waves run at the same time (so many on each CU), one element more, and nearly twice as many."""
    n = spans * waves * torch.cuda.get_device_properties(dev).multi_processor_count * 2048 + more
    check_against_oracle(oracle, dev, make_weight("calibrated_odd_scale", 1, n), level_bits)


@pytest.mark.parametrize("level_bits,waves", [((3, 5, 8), 20), ((3, 4, 6, 8), 20), ((3, 4, 5, 6, 8), 16), ((2, 3, 4, 5, 6, 7, 8), 12),
                                              ((1, 2, 3, 4, 5, 6, 7, 8), 20)])
def test_encode_elements_that_wait_for_their_level(oracle, dev, level_bits, waves):
    """Waves of five and six spans whose elements go to the levels by turns: spans of one level, of two, of all, so that what waits for a
    level is nothing, a few, as much as fits or more than the next has room for."""
    n = 5 * waves * torch.cuda.get_device_properties(dev).multi_processor_count * 2048 + 4099
    rng = np.random.default_rng(len(level_bits))
    top = np.array([0] + [(1 << (b - 1)) - 1 for b in level_bits])
    spans = n // 2048 + 1
    low, high = rng.integers(0, len(level_bits), size=(2, spans))
    low, high = np.where(rng.random(spans) < 0.2, 0, np.minimum(low, high)), np.maximum(low, high)
    level = (low[:, None] + rng.integers(0, 1 << 16, size=(spans, 2048), dtype=np.uint16) % (high - low + 1)[:, None]).reshape(-1)[:n]
    size = top[level] + 1 + rng.integers(0, 1 << 16, size=n, dtype=np.uint16) % (top[level + 1] - top[level]).clip(1)
    v = np.where(rng.integers(0, 2, size=n, dtype=np.int8) == 1, size, -size).clip(-127, 127)
    v[n // 2] = 127
    check_against_oracle(oracle, dev, torch.from_numpy(v.astype(np.float32) * 2.0 ** -9).bfloat16().reshape(1, n), level_bits)


def test_encode_elements_that_wait_for_their_level_of_six(oracle, dev):
    test_encode_elements_that_wait_for_their_level(oracle, dev, (3, 4, 5, 6, 7, 8), 12)


@pytest.mark.parametrize("n,top", [(3 * 8192 + 5, 8191), (3 * 8192 + 5, 3 * 8192 - 1), (3 * 8192 + 5, 3 * 8192 + 4), (16 * 512, 16 * 512 - 1),
                                   (16 * 512 + 1, 16 * 512), (32768 * 512, 32768 * 512 - 1), (32768 * 512 + 1, 32768 * 512)])
def test_encode_counts_by_groups_of_either_size(oracle, dev, n, top):
    """The largest weight in a whole or in the ragged part of the search for it; units counted 16 and 64 to a workgroup."""
    w = make_weight("calibrated_odd_scale", 1, n)
    w[0, top] = -4 * w.abs().max()
    check_against_oracle(oracle, dev, w, (3, 5, 8))


@pytest.mark.parametrize("units,of_units", [(32768, 32769), (32768, 32768), (40, 64), (20000, 32769), (16, 16)])
def test_encode_scratch_of_a_larger_weight(dev, units, of_units):
    """A scratch that the size call names for one weight is enough for smaller ones, and nothing behind it is written."""
    import ctypes as C

    from ixrun_amd import _lib

    L, levels = _lib.lib(), (3, 5, 8)
    n = units * 512
    w = make_weight("calibrated_odd_scale", 1, n).to(dev)
    need = int(L.ixh_encode_workspace_bytes(1, of_units * 512, len(levels)))
    ws = torch.full((need + 4096,), 0xA5, dtype=torch.uint8, device=dev)
    scale = torch.zeros(1, dtype=torch.bfloat16, device=dev)
    table = torch.empty(2 * (units + 1), dtype=torch.int32, device=dev)
    bits = (C.c_int32 * len(levels))(*levels)
    _lib.check(L.ixh_encode_scan(w.data_ptr(), 1, n, len(levels), bits, scale.data_ptr(), table.data_ptr(), ws.data_ptr(), need,
                                 _lib.current_stream(dev)))
    assert bool((ws[need:] == 0xA5).all())
    packed, whole, _ = _lib.encode_device(w, levels)
    assert torch.equal(table.view(2, -1), whole.view(2, -1))


SCAN = "ixh_encode_scan_counts"


@pytest.fixture(params=["native", "python"])
def watched_encode(request, monkeypatch, dev):
    """``encode_device`` by its native and its Python way, with what the scan's launch does on the way in ``launches``."""
    import ctypes as C

    from ixrun_amd import _lib

    L, launches = _lib.lib(), []
    scan = getattr(L, SCAN)
    proto = C.CFUNCTYPE(C.c_int, *(C.c_void_p if t is C.POINTER(C.c_int32) else t for t in scan.argtypes))
    raw = proto(C.cast(scan, C.c_void_p).value)

    def watch(*args):
        launches.append(SCAN)
        return raw(*args)

    if request.param == "native":
        watched = proto(watch)
        monkeypatch.setattr(_lib, "_native", None)
        with monkeypatch.context() as during:
            during.setattr(L, SCAN, watched)
            _lib.host()
    else:
        real = _lib.host()

        class Host:
            describe = staticmethod(real.describe)
            encode = staticmethod(lambda *a: None)

        monkeypatch.setattr(_lib, "host", lambda: Host)
        monkeypatch.setattr(L, SCAN, lambda *a: (launches.append(SCAN), scan(*a))[1])
    yield request.param, launches
    monkeypatch.undo()
    _lib._native = None  # bound to the library's own entry points again at its next use
    _lib.host()


def test_memory_for_the_bitmap_is_found_before_anything_runs(watched_encode, dev):
    """The scan writes the counts to pinned memory that an exception would give back: where memory is short for the first
    bitmap, the call fails with nothing launched."""
    from ixrun_amd import _lib

    _, launches = watched_encode
    w = torch.zeros(16384, 16384, dtype=torch.bfloat16, device=dev)  # bitmap 34 MB; rank table and scratch 4 MB
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 30 * 2 ** 20) / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            _lib.encode_device(w, (3, 5, 8))
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert not launches
    _, _, counts = _lib.encode_device(w, (3, 5, 8))
    assert launches and counts == [w.numel(), 0, 0]


@pytest.mark.parametrize("watched_encode", ["python"], indirect=True)
def test_interrupt_waits_for_the_scan(monkeypatch, watched_encode, dev):
    """An exception between the scan's launch and the counts' arrival (the Python way; the native one has no such place)
    leaves only when the stream is done with the counts' memory."""
    from ixrun_amd import _lib

    _, launches = watched_encode

    def interrupted(*args):
        raise KeyboardInterrupt

    monkeypatch.setattr(_lib.lib(), "ixh_encode_wait", interrupted)
    w = outlier_weight(512, 2048, seed=1).to(dev)
    torch.cuda.synchronize()
    torch.cuda._sleep(50_000_000)  # some 20 ms of other work in front
    assert not torch.cuda.current_stream().query()
    with pytest.raises(KeyboardInterrupt):
        _lib.encode_device(w, (3, 5, 8))
    assert launches and torch.cuda.current_stream().query()
