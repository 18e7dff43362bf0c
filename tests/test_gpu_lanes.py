"""The lane layout (``ixh_lanes_*``) through the C ABI: products of 1 to 16 activation rows against the fp64 oracle.

Shapes sit at the edges of the layout (row quads, 16-row blocks, 512-column cells, the 32768-column segments of the
list), mixes at every width of the plane, with no listed element, with rows of listed elements only, and with one row
far fuller than the others of its quad."""
import ctypes as C
import weakref

import numpy as np
import pytest
import torch

from helpers import activations, bf16_bits, bits_to_bf16, int8_mix, packed_from_int8, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    return torch.device("cuda:0")


def values(kind, out_f, in_f):
    """(int8 values, scheme, width of the plane)"""
    n = out_f * in_f
    if kind == "narrow":
        return int8_mix("only_l1", n, seed=1), (3, 5, 8), 3
    if kind == "rare":
        return int8_mix("rare_other", n, seed=1), (3, 5, 8), 3
    if kind == "four":
        v = int8_mix("only_l1", n, seed=2) * 2
        v[::67] = 100
        return v.astype(np.int8), (4, 8), 4
    if kind == "real":
        rng = np.random.default_rng(3)
        v = rng.integers(-15, 16, size=n)
        hit = rng.random(n) < 0.05
        v[hit] = rng.integers(16, 128, size=n)[hit] * (rng.integers(0, 2, size=n)[hit] * 2 - 1)
        return v.astype(np.int8), (3, 4, 5, 6, 8), 5
    if kind == "full_row":  # a quad of rows one of which is listed throughout
        v = int8_mix("no_l3", n, seed=4).reshape(out_f, in_f)
        v[out_f // 2] = 77
        return v.reshape(-1), (3, 5, 8), 5 if out_f >= 16 else 8  # (8: shorter than the list would be)
    return int8_mix("only_l3", n, seed=5), (3, 5, 8), 8


def lay_out_values(p, out_f, in_f, dev):
    from ixrun_amd import _lib
    from ixrun_amd.fused import pick_unit

    dp = _lib.DevicePacked.from_dict(p, dev)
    unit = pick_unit(in_f)
    return p, _lib.LanePacked.build(dp, dp.prefix_build(unit), unit, p["counts"])


def lay_out(kind, out_f, in_f, dev):
    v, scheme, bits = values(kind, out_f, in_f)
    p, lanes = lay_out_values(packed_from_int8(v, out_f, in_f, level_bits=scheme), out_f, in_f, dev)
    assert lanes.bits == bits
    return p, lanes


def product(lanes, x, out_f, in_f, bias=None):
    from ixrun_amd import _lib

    m = x.shape[0]
    need = lanes.gemv_workspace_bytes(m)
    ws = torch.full((need // 4 + 1,), float("nan"), dtype=torch.float32, device=x.device)
    y = torch.full((m, out_f), 7.0, dtype=torch.bfloat16, device=x.device)
    _lib.check(_lib.lib().ixh_lanes_gemv(C.byref(lanes.struct), x.data_ptr(), x.stride(0), bias.data_ptr() if bias is not None else None,
                                         m, y.data_ptr(), out_f, ws.data_ptr(), need, _lib.current_stream(x.device)))
    return y


def lib_gemv():
    from ixrun_amd import _lib

    return _lib.lib().ixh_gemv


def check(oracle, p, x, y, bias=None, once=False):
    want = oracle.gemm_f64(oracle.decode_packed_bf16(p), bf16_bits(x)).astype(np.float32)
    if once and bias is not None:
        want += bias.float().cpu().numpy()[None, :]
    want = oracle.f32_to_bf16_bits(want)
    if bias is not None and not once:
        want = oracle.f32_to_bf16_bits(oracle.bf16_bits_to_f32(want) + bias.float().cpu().numpy()[None, :])
    got = oracle.bf16_bits_to_f32(bf16_bits(y)).astype(np.float64)
    assert rel_l2(got, oracle.bf16_bits_to_f32(want)) <= 1e-3


@pytest.mark.parametrize("kind", ["narrow", "rare", "four", "real", "full_row", "wide"])
@pytest.mark.parametrize("out_f,in_f", [(16, 512), (5, 511), (67, 1003), (130, 2560), (33, 4104)])
def test_products(oracle, dev, kind, out_f, in_f):
    p, lanes = lay_out(kind, out_f, in_f, dev)
    for m in (1, 2, 3, 4, 5, 8, 9, 16):
        x = activations(m, in_f, seed=m)
        y = product(lanes, x.to(dev), out_f, in_f)
        check(oracle, p, x, y)
        assert torch.equal(y, product(lanes, x.to(dev), out_f, in_f))  # the order of the sums is fixed


@pytest.mark.parametrize("kind", ["rare", "real"])
@pytest.mark.parametrize("out_f,in_f", [(6, 33800), (4100, 520)])
def test_long_rows_and_many_rows(oracle, dev, kind, out_f, in_f):
    """More columns than a segment of the list; more row blocks than a workgroup has waves."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    for m in (1, 2, 4, 16):
        x = activations(m, in_f, seed=m)
        check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))


@pytest.mark.parametrize("out_f,in_f,m", [(32801, 25, 9), (32801, 25, 16), (16501, 1030, 9), (16501, 1030, 16)])
def test_four_bits_by_the_larger_table(oracle, dev, out_f, in_f, m):
    """Nine to sixteen rows of more than 32 cells a CU: sixteen copies of the pair table beside the activations."""
    p, lanes = lay_out("four", out_f, in_f, dev)
    x = activations(m, in_f, seed=m)
    check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))


@pytest.mark.parametrize("at", [5, 32767, 32768, 33799])
@pytest.mark.parametrize("listed", [1, 16, 17, 33])
def test_list_of_one_segment_of_long_rows(oracle, dev, at, listed):
    """The other segment of the rows has nothing listed; the last group ends with the segment or behind it."""
    out_f, in_f = 1028, 33800  # 257 row quads: two a workgroup
    v = int8_mix("only_l1", out_f * in_f, seed=6).reshape(out_f, in_f)
    first = min(at, in_f - 4 * listed) if at != 32767 else 32768 - 4 * listed
    v[:, first : first + 4 * listed : 4] = 90
    p, lanes = lay_out_values(packed_from_int8(v.reshape(-1), out_f, in_f), out_f, in_f, dev)
    assert lanes.bits == 3
    for m in (1, 2):
        x = activations(m, in_f, seed=m)
        check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))


@pytest.mark.parametrize("kind", ["rare", "real"])
@pytest.mark.parametrize("out_f,in_f,m", [(1028, 37888, 2), (1025, 37380, 2), (1028, 75776, 1), (1028, 75771, 1)])
def test_rows_that_leave_no_room_for_sums_of_cells(oracle, dev, kind, out_f, in_f, m):
    """Two row quads a workgroup of as many cells as LDS holds the activations of: the waves' sums are kept instead."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    assert lanes.gemv_workspace_bytes(m) == 0
    x = activations(m, in_f, seed=m)
    check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))


@pytest.mark.parametrize("kind", ["rare", "four", "real", "full_row", "wide"])
@pytest.mark.parametrize("out_f,in_f", [(4096, 2048), (4093, 2041), (17 * 1024 - 3, 512), (8192, 2048), (8185, 2040), (8200, 2048), (40, 8192), (40, 8200)])
def test_a_cell_or_two_a_wave(oracle, dev, kind, out_f, in_f):
    """16, 17, 32 and 36 cells a workgroup, its last row quads incomplete or missing; rows of as many cells as waves and of one more."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    for m in (1, 2, 3, 4):
        x = activations(m, in_f + 8, seed=m)[:, 8 * (m % 2) :][:, :in_f]
        check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f, bias.to(dev) if m > 1 else None), bias if m > 1 else None)


@pytest.mark.parametrize("kind", ["rare", "real"])
@pytest.mark.parametrize("out_f", [63488, 70000])
def test_more_row_quads_than_a_wave_has_lanes(oracle, dev, kind, out_f):
    """62 and 69 row quads a workgroup, whose lists begin in more places than a wave looks up at once (one row; two and four of such layers
    are the other kernel's); most have one group in many row quads, or none."""
    in_f = 40
    p, lanes = lay_out(kind, out_f, in_f, dev)
    for m in (1, 2, 4):
        x = activations(m, in_f, seed=m)
        check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))
    v = int8_mix("only_l1", out_f * in_f, seed=6).reshape(out_f, in_f)
    v[-300:, 3] = 90  # all that is listed lies in a workgroup's last row quads
    p, lanes = lay_out_values(packed_from_int8(v.reshape(-1), out_f, in_f), out_f, in_f, dev)
    x = activations(1, in_f, seed=9)
    check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))


@pytest.mark.parametrize("kind", ["rare", "real"])
@pytest.mark.parametrize("out_f,in_f,m", [(16 * 257 + 3, 1030, 5), (40, 5120, 8), (40, 5121, 8), (40, 10240, 7), (37, 3584, 16), (37, 3586, 9),
                                          (20, 17407, 6), (20, 17409, 12), (3, 520, 16)])
def test_rows_at_the_edges_of_their_slices(oracle, dev, kind, out_f, in_f, m):
    """5 to 16 rows: as many columns as LDS holds and just more, a block more than there are workgroups, waves without a step,
    rows that no pair of columns divides."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    for skip in (0, 1, 2):  # whole 16-byte pieces (nine rows and more may take another way then), pairs or neither
        x = activations(m, in_f + 8, seed=m).to(dev)[:, skip : skip + in_f]
        y = product(lanes, x, out_f, in_f, bias.to(dev))
        check(oracle, p, x.cpu(), y, bias)
        assert torch.equal(y, product(lanes, x, out_f, in_f, bias.to(dev)))


@pytest.mark.parametrize("ldx", [(1 << 27) - 2, (1 << 27) - 1, 1 << 27, (1 << 27) + 2])
def test_rows_far_apart(oracle, dev, ldx):
    """Strides on both sides of 2^27 elements, up to which pairs are asked for at places in 32 bits."""
    out_f, in_f, m = 37, 3586, 16
    p, lanes = lay_out("real", out_f, in_f, dev)
    x = activations(m, in_f, seed=m)
    far = torch.empty((m - 1) * ldx + in_f, dtype=torch.bfloat16, device=dev).as_strided((m, in_f), (ldx, 1))
    far.copy_(x)
    for n in (5, 8, 16):
        check(oracle, p, x[:n], product(lanes, far[:n], out_f, in_f))


@pytest.mark.parametrize("kind", ["four", "real"])
@pytest.mark.parametrize("out_f,in_f", [(4131, 1500), (4131, 3080)])
def test_both_tables_of_pairs(oracle, dev, kind, out_f, in_f):
    """Planes of 4 and 5 bits with few and with many cells a CU: the smaller table of pairs (the other tests' too) and the larger."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    for m in (1, 2, 4, 7):
        x = activations(m, in_f, seed=m)
        check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))


@pytest.mark.parametrize("m", [1, 4, 7])
def test_bias_and_unaligned_activations(oracle, dev, m):
    out_f, in_f = 37, 1536
    p, lanes = lay_out("real", out_f, in_f, dev)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    wide = activations(m, in_f + 9, seed=3).to(dev)
    for x in (wide[:, :in_f], wide[:, 3 : 3 + in_f]):
        check(oracle, p, x.cpu(), product(lanes, x, out_f, in_f, bias.to(dev)), bias)


@pytest.mark.parametrize("kind", ["narrow", "rare", "four", "real", "full_row", "wide"])
@pytest.mark.parametrize("out_f,in_f", [(16, 512), (5, 520), (300, 1032), (67, 4104)])
def test_many_rows(oracle, dev, kind, out_f, in_f):
    """The decode into matrix-core tiles: edges of the blocks of 16 activation rows and of the groups of 128, of the blocks
    of 16 weight rows, of the 128-column stages and of the cells."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    for m in (1, 17, 33, 48, 50, 79, 96, 97, 128, 129, 300):
        wide = activations(m, in_f + 8, seed=m).to(dev)
        x, b = wide[:, 8:], bias if m % 2 else None
        y = [torch.full((m, out_f), 7.0, dtype=torch.bfloat16, device=dev) for _ in range(2)]
        for t in y:
            lanes.gemm(x, t, None if b is None else b.to(dev))
        check(oracle, p, x.cpu(), y[0], b, once=True)
        assert torch.equal(*y)  # the order of the sums is fixed


@pytest.mark.parametrize("kind,out_f,in_f", [("rare", 24600, 1032), ("real", 8200, 3080), ("full_row", 8200, 3080), ("four", 1000, 25400),
                                             ("wide", 400, 66000)])
def test_many_rows_of_the_largest_weights(oracle, dev, kind, out_f, in_f):
    """Tiles of 128 weight rows: each width of the sums and a second group of rows; a workgroup with a whole tile, with a slice of
    one and with the end of one and the start of the next; lists longer than are held; y's rows at odd multiples of 2 bytes."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    wide = activations(513, in_f + 8, seed=3).to(dev)
    x = wide[:, 8:]
    weight = bits_to_bf16(oracle.decode_packed_bf16(p)).to(dev).reshape(out_f, in_f).float()
    exact = x.float() @ weight.t()
    for m in (129, 200, 257, 500, 513):
        b = bias if m % 2 else None
        want = (exact[:m] if b is None else exact[:m] + b.to(dev).float()).bfloat16()
        y = torch.full((2, m, out_f + m % 3), 7.0, dtype=torch.bfloat16, device=dev)
        for t in y:
            lanes.gemm(x[:m], t[:, :out_f], None if b is None else b.to(dev))
        # both are one rounding to bf16 of sums whose fp32 errors are far below it: they differ where a sum is next to a tie
        assert rel_l2(y[0, :, :out_f].float().cpu().numpy(), want.float().cpu().numpy()) <= 1e-3
        assert torch.equal(y[0], y[1]) and (y[:, :, out_f:] == 7).all()


@pytest.mark.parametrize("kind,out_f,in_f", [("rare", 65536, 520), ("four", 70000, 400), ("real", 8200, 3080), ("four", 1000, 25400)])
def test_scratch_of_prompts_at_any_address(oracle, dev, kind, out_f, in_f):
    """Two whole tiles a workgroup (no sums in memory), more tiles than workgroups and shared ones, fewer shared, and several
    workgroups to a tile: as many bytes as are asked for, at an odd address, hold all that is written."""
    from ixrun_amd import _lib

    p, lanes = lay_out(kind, out_f, in_f, dev)
    weight = bits_to_bf16(oracle.decode_packed_bf16(p)).to(dev).reshape(out_f, in_f).float()
    for m in (130, 513):
        x = activations(m, in_f, seed=m).to(dev)
        need = lanes.gemm_workspace_bytes(m)
        ws = torch.full((need + 256,), 0xA5, dtype=torch.uint8, device=dev)
        y = torch.full((m, out_f), 7.0, dtype=torch.bfloat16, device=dev)
        _lib.check(_lib.lib().ixh_lanes_gemm(C.byref(lanes.struct), x.data_ptr(), in_f, None, m, y.data_ptr(), out_f, ws.data_ptr() + 101,
                                             need, _lib.current_stream(dev)))
        assert bool((ws[:101] == 0xA5).all()) and bool((ws[101 + need :] == 0xA5).all())
        want = (x.float() @ weight.t()).bfloat16()
        # (see test_many_rows_of_the_largest_weights)
        assert rel_l2(y.float().cpu().numpy(), want.float().cpu().numpy()) <= 1e-3
        again = torch.empty_like(y)
        lanes.gemm(x, again)
        assert torch.equal(y, again)


@pytest.mark.parametrize("out_f,in_f,m", [(4100, 520, 20), (4500, 1536, 130), (20, 33800, 40)])
def test_many_rows_of_larger_weights(oracle, dev, out_f, in_f, m):
    """Several blocks of weight rows a workgroup, and slices of several cells."""
    p, lanes = lay_out("real", out_f, in_f, dev)
    x = activations(m, in_f, seed=m)
    y = torch.full((m, out_f), 7.0, dtype=torch.bfloat16, device=dev)
    lanes.gemm(x.to(dev), y)
    check(oracle, p, x, y)


@pytest.mark.parametrize("kind,out_f,in_f", [("real", 4347, 6032), ("real", 5120, 5120), ("rare", 1024, 8192), ("four", 1000, 4096)])
def test_scratch_of_any_count_up_to_sixteen(oracle, dev, kind, out_f, in_f):
    """What five rows ask for is enough for any count up to sixteen, whichever kernel takes it, and nothing behind it is written."""
    from ixrun_amd import _lib

    p, lanes = lay_out(kind, out_f, in_f, dev)
    need = lanes.gemv_workspace_bytes(5)
    assert all(lanes.gemv_workspace_bytes(m) == need for m in range(5, 17))
    ws = torch.full((need + 4096,), 0xA5, dtype=torch.uint8, device=dev)
    weight = bits_to_bf16(oracle.decode_packed_bf16(p)).to(dev).reshape(out_f, in_f).float()
    for m in range(5, 17):
        x = activations(m, in_f, seed=m).to(dev)
        y = torch.full((m, out_f), 7.0, dtype=torch.bfloat16, device=dev)
        _lib.check(_lib.lib().ixh_lanes_gemv(C.byref(lanes.struct), x.data_ptr(), in_f, None, m, y.data_ptr(), out_f, ws.data_ptr(), need,
                                             _lib.current_stream(dev)))
        # (see test_many_rows_of_the_largest_weights)
        assert rel_l2(y.float().cpu().numpy(), (x.float() @ weight.t()).bfloat16().float().cpu().numpy()) <= 1e-3
    assert bool((ws[need:] == 0xA5).all())


def planned(bounds, dev, out_f, in_f, m):
    """(groups of activation rows, blocks of 16 of them in a group, slices of the columns, groups of weight rows) of k_lanes_gemm."""
    out = (C.c_uint32 * 4)()
    bounds.plan(out_f, -(-in_f // 512), m, torch.cuda.get_device_properties(dev).multi_processor_count, out)
    return tuple(out)


@pytest.mark.parametrize("kind,out_f,in_f,m,most,least", [
    ("real", 13616, 2560, 1, 17, 16), ("rare", 16400, 512, 512, 29, 28), ("real", 9808, 6656, 17, 33, 32),
    ("rare", 9984, 6656, 17, 33, 32), ("four", 10048, 6656, 17, 34, 33)])
def test_workgroups_of_several_rounds(bounds, dev, oracle, kind, out_f, in_f, m, most, least):
    """More blocks of weight rows than a workgroup has waves, and one more for some than for others: also where these have a round less."""
    groups, blocks = planned(bounds, dev, out_f, in_f, m)[3], -(-out_f // 16)
    assert (-(-blocks // groups), blocks // groups) == (most, least) or torch.cuda.get_device_properties(dev).multi_processor_count != 256
    p, lanes = lay_out(kind, out_f, in_f, dev)
    x = activations(m, in_f, seed=m).to(dev)
    weight = bits_to_bf16(oracle.decode_packed_bf16(p)).to(dev).reshape(out_f, in_f).float()
    y = torch.full((m, out_f), 7.0, dtype=torch.bfloat16, device=dev)
    lanes.gemm(x, y)
    # (see test_many_rows_of_the_largest_weights)
    assert rel_l2(y.float().cpu().numpy(), (x.float() @ weight.t()).bfloat16().float().cpu().numpy()) <= 1e-3


@pytest.mark.parametrize("kind,out_f,in_f", [("rare", 1638, 2560), ("rare", 1639, 2560), ("real", 40, 2040), ("real", 40, 2048),
                                             ("real", 4095, 2048), ("real", 4096, 2048), ("four", 5120, 5112), ("four", 5120, 5120),
                                             ("real", 5120, 5112), ("real", 5120, 5120), ("wide", 5120, 5112), ("wide", 5120, 5120),
                                             ("real", 9420, 5120), ("real", 9421, 5120), ("wide", 7782, 5120), ("wide", 7783, 5120)])
def test_nine_to_sixteen_rows_either_way(oracle, dev, kind, out_f, in_f):
    """Weights on both sides of the lines between the two kernels that take nine to sixteen rows; few blocks and many, one cell to ten a slice."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    for m in (9, 16):
        x = activations(m, in_f, seed=m)
        check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f, bias.to(dev)), bias)


# rows of activations that one workgroup takes, 16 a block: a shape whose cut leaves them together (33 slices, three or four blocks of weight
# rows a workgroup and one less; the last cell and its last 128 columns incomplete)
def shape_of_blocks(bounds, dev, m):
    out_f, in_f = 205 if m <= 48 else 397, 16800
    together = planned(bounds, dev, out_f, in_f, m)[1] == max(-(-m // 16), 1)
    assert together or torch.cuda.get_device_properties(dev).multi_processor_count != 256
    return out_f, in_f


@pytest.mark.parametrize("m", [1, 16, 17, 32, 33, 48, 50, 64, 65, 79, 81, 96, 97, 112, 113, 127, 128])
@pytest.mark.parametrize("kind", ["narrow", "rare", "four", "real", "full_row", "wide"])
def test_each_count_of_blocks_of_activation_rows(bounds, oracle, dev, kind, m):
    """Every form of the kernel, with whole and nearly empty last blocks."""
    out_f, in_f = shape_of_blocks(bounds, dev, m)
    p, lanes = lay_out(kind, out_f, in_f, dev)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16().to(dev) if m % 2 else None
    x = activations(m, in_f + 8, seed=m).to(dev)[:, 8:]
    weight = bits_to_bf16(oracle.decode_packed_bf16(p)).to(dev).reshape(out_f, in_f).double()
    y = torch.full((2, m, out_f), 7.0, dtype=torch.bfloat16, device=dev)
    for t in y:
        lanes.gemm(x, t, bias)
    want = (x.double() @ weight.t() + (0 if bias is None else bias.double())).float().bfloat16()
    # (see test_many_rows_of_the_largest_weights)
    assert rel_l2(y[0].float().cpu().numpy(), want.float().cpu().numpy()) <= 1e-3
    assert torch.equal(y[0], y[1])


@pytest.mark.parametrize("scale", [2.0 ** -100, 1.5 * 2.0 ** 99, 2.0 ** 100, 1.75 * 2.0 ** 112, 2.0 ** 120])
@pytest.mark.parametrize("kind", ["four", "real"])
def test_many_rows_at_extreme_scales(bounds, oracle, dev, kind, scale):
    """Multiples of the scale by up to 2^20 stand behind codes of five bits; from 2^100 on they would be infinities.  Every count of blocks of
    16 activation rows, and nine and 16 as a batch (rounded before the bias as well as after it)."""
    down = 2.0 ** -int(np.log2(scale))  # (a power of two takes the sums to where their squares are finite; it changes no rounding)
    for m in (9, 16, 17, 48, 64, 80, 96, 112, 128):
        out_f, in_f = shape_of_blocks(bounds, dev, m)
        v, scheme, _ = values(kind, out_f, in_f)
        p = packed_from_int8(v, out_f, in_f, level_bits=scheme)
        p["scale"] = torch.full_like(p["scale"], scale)
        p, lanes = lay_out_values(p, out_f, in_f, dev)
        x = (activations(m, in_f, seed=m).float() * 2.0 ** -12).bfloat16().to(dev)
        weight = bits_to_bf16(oracle.decode_packed_bf16(p)).to(dev).reshape(out_f, in_f).double()
        want = (x.double() @ weight.t() * down).float().bfloat16()
        if m <= 16:
            bias = (want[0].double() / down).bfloat16()
            y = product(lanes, x, out_f, in_f, bias)
            want = (want.double() + bias.double() * down).float().bfloat16()
        else:
            y = torch.full((m, out_f), 7.0, dtype=torch.bfloat16, device=dev)
            lanes.gemm(x, y)
        assert bool(y.isfinite().all())
        assert rel_l2((y.double() * down).cpu().numpy(), want.double().cpu().numpy()) <= 1e-3


@pytest.mark.parametrize("scale,lanes", [(2.0 ** 121, True), ((1 + 2.0 ** -7) * 2.0 ** 121, False), (float("inf"), False), (float("nan"), False)])
def test_weights_that_round_to_infinities(oracle, dev, scale, lanes):
    """The layout is made from the bf16 weights and has no place for an infinite one: such a layer (its largest weight is the largest bf16
    value) has none, also when its state comes later, and its products have the infinities of its decode."""
    from ixrun_amd.engine import StreamingLinear

    out_f, in_f = 260, 2048
    v = values("rare", out_f, in_f)[0]
    v[5::1009] = 127 - 254 * (np.arange(v[5::1009].size) % 2)
    p = packed_from_int8(v, out_f, in_f)
    other = StreamingLinear(p, None)
    assert other._lanes is not None
    p = dict(p, scale=torch.full_like(p["scale"], scale))
    layer = StreamingLinear(p, None)
    other.load_state_dict(layer.state_dict())
    weight = bits_to_bf16(oracle.decode_packed_bf16(p)).reshape(out_f, in_f).double()
    assert bool(weight.isfinite().all()) == lanes
    for each in (layer, other):
        assert (each._lanes is not None) == lanes
        each._set_shared_buf(torch.empty(out_f * in_f, dtype=torch.bfloat16, device=dev))
        for m in (1, 2, 4, 8, 16, 17, 100):
            x = (activations(m, in_f, seed=m).float() * 2.0 ** -20).bfloat16()
            with torch.no_grad():
                y = each(x.to(dev)).double().cpu()
            want = x.double() @ weight.t()
            assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y[y.isinf()], want[want.isinf()])
            fine = want.isfinite()  # (the power of two takes the squares to where they are finite; it changes no rounding)
            assert rel_l2(y[fine].numpy() * 2.0 ** -110, want[fine].bfloat16().double().numpy() * 2.0 ** -110) <= 1e-3 or not fine.any()


def test_prompts_of_a_layer_take_the_lanes_in_every_form(oracle, dev):
    """What goes to the fused decode+GEMM comes out as from the layer without lanes, whatever the activations' form; what it
    is not for (gradients, other types, more rows) still goes through the decode."""
    from ixrun_amd.engine import StreamingLinear

    out_f, in_f = 520, 1032
    v, scheme, _ = values("real", out_f, in_f)
    p = packed_from_int8(v, out_f, in_f, level_bits=scheme)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    layer, plain = StreamingLinear(p, bias=bias), StreamingLinear(p, bias=bias, lanes=False)
    bufs = [torch.zeros(p["N"], dtype=torch.bfloat16, device=dev) for _ in range(2)]
    for one, buf in zip((layer, plain), bufs):
        one._set_shared_buf(buf)
    wide = activations(160, in_f + 3, seed=5).to(dev)
    flat = wide.reshape(-1)[3 : 3 + 40 * in_f]  # contiguous, 6 bytes off
    forms = [wide[:17, :in_f], wide[:, 3:], wide[:33, :in_f].reshape(3, 11, in_f), flat.view(4, 10, in_f), wide[:1, :in_f].expand(20, in_f),
             wide[:, :in_f].t().contiguous().t(), wide[::2, :in_f]]
    for x in forms:
        got, want = layer(x), plain(x)
        assert got.shape == want.shape and got.dtype == want.dtype and got.is_contiguous()
        # the library may round its product before it adds the bias: half a bf16 step more on either side
        assert rel_l2(got.double().cpu().numpy(), want.double().cpu().numpy()) <= 2 ** -8
        check(oracle, p, x.reshape(-1, in_f).cpu(), got.reshape(-1, out_f), bias, once=True)
    assert not bool(bufs[0].any())
    graph, x = torch.cuda.CUDAGraph(), wide[:50, :in_f].contiguous()
    layer(x)
    with torch.cuda.graph(graph):
        y = layer(x)
    for seed in (1, 2, 3):
        x.copy_(activations(50, in_f, seed=seed))
        graph.replay()
        assert torch.equal(y, layer(x))
    assert not bool(bufs[0].any())
    x = wide[:40, :in_f].contiguous().requires_grad_()
    assert layer(x).requires_grad and bool(bufs[0].any())
    many = activations(600, in_f, seed=6).to(dev)
    for x in (many, wide[:40, :in_f].float()):
        assert rel_l2(layer(x).double().cpu().numpy(), plain(x).double().cpu().numpy()) <= 1e-3


@pytest.mark.parametrize("kind,out_f,in_f", [(k, 67, 1000) for k in ("narrow", "rare", "four", "real", "full_row", "wide")] +
                         [("real", 9, 511), ("real", 6000, 1032), ("rare", 6, 32000), ("real", 6, 32768), ("real", 6, 33800)])
def test_infinite_activations(oracle, dev, kind, out_f, in_f):
    """An infinite activation gives an infinity of the right sign, or NaN where a row's own weight is zero or another
    infinity meets it: where the list's padding points (column 0), in columns with listed elements and in others."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    w = bits_to_bf16(oracle.decode_packed_bf16(p)).reshape(out_f, in_f).double()
    listed = w.abs().argmax(1)  # of each row: the columns its largest weights are in
    for m in (1, 2, 3, 4, 8, 20):
        if m > 16 and in_f % 8:
            continue
        x = activations(m, in_f, seed=m)
        for j in range(m):
            x[j, (0, int(listed[j % out_f]), in_f - 1, int(listed[(j + 1) % out_f]))[j % 4]] = float("inf") if j % 3 else -float("inf")
        if m > 2:
            x[2, int(listed[2])] = float("inf")  # a second one
            x[m - 1, 5] = float("nan")
        want = torch.stack([(w * x[j].double()).sum(1) for j in range(m)])
        if m <= 16:
            y = product(lanes, x.to(dev), out_f, in_f).cpu().double()
        else:
            y = torch.empty((m, out_f), dtype=torch.bfloat16, device=dev)
            lanes.gemm(x.to(dev), y)
            y = y.cpu().double()
        assert bool(want.isinf().any())
        assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y[y.isinf()], want[want.isinf()])
        fine = want.isfinite()
        assert rel_l2(y[fine].numpy(), want[fine].bfloat16().double().numpy()) <= 1e-3


def with_infinities(x, w):
    """In two of three rows an infinity or two, in some a NaN: in columns where a weight row has its largest weight (a listed one, where it
    has any), in the first and last column, and in the first and last rows of the blocks of 16."""
    m, in_f = x.shape
    for j in range(m):
        if j % 3 == 1:
            continue
        largest = int(w[j % w.shape[0]].abs().argmax())
        x[j, (0, largest, in_f - 1, in_f // 2)[j % 4]] = float("inf") if j % 5 else -float("inf")
        if j % 4 == 2:
            x[j, largest] = -float("inf")
        if j % 7 == 3:
            x[j, 5] = float("nan")
    x[m - 1, in_f - 1] = float("inf")
    return x


def same_infinities(y, want):
    y, want = y.double().cpu(), want.cpu()
    assert bool(want.isinf().any()) and bool(want.isfinite().any())
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y[y.isinf()], want[want.isinf()])
    fine = want.isfinite()
    assert rel_l2(y[fine].numpy(), want[fine].bfloat16().double().numpy()) <= 1e-3


@pytest.mark.parametrize("kind", ["narrow", "rare", "four", "real", "full_row", "wide"])
@pytest.mark.parametrize("out_f,in_f", [(67, 1000), (37, 1900), (20, 8003)])
def test_infinite_activations_of_nine_to_sixteen_rows(oracle, dev, kind, out_f, in_f):
    """As test_infinite_activations, where the kernel keeps sixteen rows of a column together (rows of one cell's and a few cells'
    columns, and longer ones of no whole pieces, which no other kernel takes)."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    w = bits_to_bf16(oracle.decode_packed_bf16(p)).reshape(out_f, in_f).double()
    for m in (9, 16):
        x = with_infinities(activations(m, in_f, seed=m), w)
        same_infinities(product(lanes, x.to(dev), out_f, in_f), torch.stack([(w * row.double()).sum(1) for row in x]))


@pytest.mark.parametrize("kind,out_f,in_f", [("rare", 24600, 1032), ("real", 8200, 3080), ("full_row", 8200, 3080), ("four", 1000, 25400),
                                             ("wide", 400, 66000)])
def test_infinite_activations_of_large_prompts(oracle, dev, kind, out_f, in_f):
    """The same through the tiles of 128 weight rows: each width of the sums, and a second group of rows."""
    p, lanes = lay_out(kind, out_f, in_f, dev)
    w = bits_to_bf16(oracle.decode_packed_bf16(p)).to(dev).reshape(out_f, in_f).double()
    for m in (129, 300, 520):
        x = with_infinities(activations(m, in_f, seed=m).to(dev), w)
        y = torch.full((m, out_f), 7.0, dtype=torch.bfloat16, device=dev)
        lanes.gemm(x, y)
        same_infinities(y, x.double() @ w.t())


@pytest.mark.parametrize("in_f", [1, 3, 7, 8, 9, 15])
def test_rows_of_a_few_columns(oracle, dev, in_f):
    """Rows shorter than, as long as and just longer than a 16-byte piece."""
    out_f = 21
    p, lanes = lay_out("rare", out_f, in_f, dev)
    for m in (1, 2, 4, 6):
        x = activations(m, in_f, seed=m)
        check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))


@pytest.mark.parametrize("listed", [0, 63, 64, 65, 128])
def test_list_that_ends_on_a_whole_group(oracle, dev, listed):
    """All listed elements in the first cells of a tensor: what is behind them starts at the list's end, which at 64 and 128
    is the end of its last group as well."""
    out_f, in_f = 260, 1536
    v = int8_mix("only_l1", out_f * in_f, seed=6).reshape(out_f, in_f)
    v[0, 7 : 7 + 2 * listed : 2] = 90
    p = packed_from_int8(v.reshape(-1), out_f, in_f)
    _, lanes = lay_out_values(p, out_f, in_f, dev)
    assert lanes.bits == 3 and int(lanes.tensors[1][-1]) == listed
    groups = max(-(-listed // 64), 1)
    lanes.struct.n_quads = 64 * groups  # (no room behind the last group that the list needs)
    for m in (1, 2, 4, 8):
        x = activations(m, in_f, seed=m)
        check(oracle, p, x, product(lanes, x.to(dev), out_f, in_f))


@pytest.mark.parametrize("kind", ["rare", "real"])
def test_prompts_from_native_code(dev, kind):
    """17 rows up to the last count that the lanes are the fastest way for: the same bits as by Python's way, and left to it where
    they always were (more rows, views, odd addresses, gradients, autocast to another type, a switch turned off)."""
    from ixrun_amd.engine import StreamingLinear

    out_f, in_f = 1030, 1024
    v, scheme, _ = values(kind, out_f, in_f)
    p = packed_from_int8(v, out_f, in_f, level_bits=scheme)
    layer, other = StreamingLinear(p, bias := torch.randn(out_f).bfloat16()), StreamingLinear(p, bias)
    other._native = None
    most = layer._native.many_rows
    assert layer._lanes_gemm_wins(most) and not layer._lanes_gemm_wins(most + 1)
    wide = activations(most + 2, in_f + 8, seed=3).to(dev)

    def same(x, native):
        assert (layer._native.many(x) is not None) == native
        y = layer(x)
        assert torch.equal(y, other(x)) and y.shape == x.shape[:-1] + (out_f,)

    for rows in (16, 17, 33, most, most + 1):
        same(wide[:rows, :in_f].contiguous(), 17 <= rows <= most)
    x = wide[:40, :in_f].contiguous()
    same(x.view(5, 8, in_f), True)
    same(x.view(2, 20, 1, in_f).transpose(0, 1), False)
    same(wide.view(-1)[1 : 1 + 40 * in_f].view(40, in_f), False)
    assert layer._native.many(x.clone().requires_grad_()) is None and layer._native.many(x.float()) is None
    with torch.autocast("cuda", dtype=torch.float16):
        assert layer._native.many(x) is None
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = layer(x)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(y, other(x))
    layer._set_shared_buf(torch.zeros(p["N"], dtype=torch.bfloat16, device=dev))
    layer(x)
    assert not bool(layer._w_buf.any())
    layer._gemm_ok = False
    layer(x)
    assert bool(layer._w_buf.any())


@pytest.mark.parametrize("kind,out_f,in_f,most", [
    ("real", 1020, 1024, 1024), ("listed", 1023, 1024, 1024), ("real", 1030, 1024, 512), ("listed", 1030, 1024, 256), ("rare", 8192, 1024, 512),
    ("rare", 8193, 520, 256), ("four", 4099, 2048, 256), ("four", 4099, 4096, 256), ("wide", 6001, 4192, 256),
    ("wide", 6004, 4192, 512)])
def test_how_many_rows_the_lanes_serve(dev, kind, out_f, in_f, most):
    """The last prompt that goes to the lanes, on both sides of each bound (weights, listed elements, rows of weights): there and
    one row further the layer's result is the decoded weight's product, whichever way it goes."""
    from ixrun_amd.engine import StreamingLinear

    v, scheme, _ = values("four" if kind == "listed" else kind, out_f, in_f)
    if kind == "listed":
        v[::11] = 100
    p = packed_from_int8(v, out_f, in_f, level_bits=scheme)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    layer = StreamingLinear(p, bias=bias)
    assert layer._native.many_rows == most
    wide = activations(most + 1, in_f, seed=4).to(dev)
    layer._set_shared_buf(torch.zeros(p["N"], dtype=torch.bfloat16, device=dev))
    weight = layer._decode().float()
    for rows in (most - 15, most, most + 1):
        x = wide[:rows]
        y = layer(x)
        assert (layer._native.many(x) is not None) == (rows <= most)
        # one rounding to bf16 of sums whose fp32 errors are far below it, and the same of the general path's
        assert rel_l2(y.float().cpu().numpy(), (x.float() @ weight.t() + bias.to(dev).float()).bfloat16().float().cpu().numpy()) <= 1e-3
        assert rel_l2(y.float().cpu().numpy(), layer._decode_and_multiply(x).float().cpu().numpy()) <= 2e-3


@pytest.mark.parametrize("first", ["short", "long"])
def test_prompts_go_by_the_list_that_is_loaded(dev, first):
    """Which prompts the lanes serve follows from the elements listed now, not from the memory that an earlier list of the layer left: a
    layer that has loaded a state goes the way of a new one of it."""
    from ixrun_amd.engine import StreamingLinear

    out_f, in_f, listed = 2048, 1024, 43
    lists = {}
    for kind in ("short", "long"):  # equal level counts: the elements of a quad's four rows, or four times as many of one of them
        v = values("four", out_f, in_f)[0].reshape(out_f, in_f)
        v[v == 100] = 6
        if kind == "short":
            v[:, : 16 * listed : 16] = 100
        else:
            v[::4, : 16 * listed : 4] = 100
        lists[kind] = packed_from_int8(v.reshape(-1), out_f, in_f, level_bits=(4, 8))
    assert lists["short"]["counts"] == lists["long"]["counts"]
    fresh = {kind: StreamingLinear(p) for kind, p in lists.items()}
    layer = StreamingLinear(lists[first])
    buf = torch.zeros(out_f * in_f, dtype=torch.bfloat16, device=dev)
    for each in (layer, *fresh.values()):
        each._set_shared_buf(buf)
    x = activations(512, in_f, seed=3).to(dev)
    for kind in ("long", "short", "long", "short", "short"):
        layer.load_state_dict(fresh[kind].state_dict())
        assert layer._native.many_rows == fresh[kind]._native.many_rows == {"short": 512, "long": 256}[kind]
        for rows in (256, 257, 512):
            assert layer._lanes_gemm_wins(rows) == fresh[kind]._lanes_gemm_wins(rows) == (rows <= layer._native.many_rows)
            assert torch.equal(layer(x[:rows]), fresh[kind](x[:rows]))


@pytest.mark.parametrize("kind,out_f,in_f", [("rare", 24600, 1032), ("real", 8200, 3080)])
def test_large_prompts_of_a_layer(oracle, dev, kind, out_f, in_f):
    """Prompts of a layer large enough for tiles of 128 weight rows, with a bias: from native code, from Python, as views, and
    replayed from a graph between eager calls; the decode buffer stays untouched."""
    from ixrun_amd.engine import StreamingLinear

    v, scheme, _ = values(kind, out_f, in_f)
    p = packed_from_int8(v, out_f, in_f, level_bits=scheme)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    layer, python = StreamingLinear(p, bias=bias), StreamingLinear(p, bias=bias)
    python._native = None
    buf = torch.zeros(p["N"], dtype=torch.bfloat16, device=dev)
    layer._set_shared_buf(buf)
    python._set_shared_buf(buf)
    assert layer._native.many_rows == 512
    weight = bits_to_bf16(oracle.decode_packed_bf16(p)).to(dev).reshape(out_f, in_f).float()
    wide = activations(512, in_f + 8, seed=3).to(dev)
    for rows in (129, 300, 512):
        x = wide[:rows, :in_f].contiguous()
        assert layer._native.many(x) is not None
        y = layer(x)
        # one rounding to bf16 of sums whose fp32 errors are far below it
        assert rel_l2(y.float().cpu().numpy(), (x.float() @ weight.t() + bias.to(dev).float()).bfloat16().float().cpu().numpy()) <= 1e-3
        assert torch.equal(y, python(x)) and torch.equal(y, layer(wide[:rows, :in_f]))
        assert torch.equal(y, layer(x.view(1, rows, in_f))[0])
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            z = layer(x)
        for seed in (1, 2, 3):
            x.copy_(activations(rows, in_f, seed=seed))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(z, layer(x))
    assert not bool(buf.any())


@pytest.mark.parametrize("native", [True, False])
def test_prompts_without_room_for_their_sums_take_the_decode_buffer(oracle, dev, native):
    """Where the allocator has no room for a prompt's sums (here: a limit on this process) a layer with a decode buffer is served
    from that, and one without raises."""
    from ixrun_amd.engine import StreamingLinear

    out_f, in_f, rows = 1000, 25400, 400
    v, scheme, _ = values("four", out_f, in_f)
    p = packed_from_int8(v, out_f, in_f, level_bits=scheme)
    bias = (torch.randn(out_f, generator=torch.Generator().manual_seed(1)) * 0.5).bfloat16()
    layer = StreamingLinear(p, bias=bias)
    if not native:
        layer._native = None
    layer._set_shared_buf(torch.zeros(p["N"], dtype=torch.bfloat16, device=dev))
    x = activations(rows, in_f, seed=3).to(dev)
    want = layer(x).clone()
    assert not bool(layer._w_buf.any())
    layer._gemm_ok = False
    layer(x)  # (the library takes its workspace now)
    layer._gemm_ok = True
    layer._w_buf.zero_()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.empty_cache()
    room = layer._lanes.gemm_workspace_bytes(rows) // 2
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(dev) + room) / total, dev)
        got = layer(x)
        assert bool(layer._w_buf.any())
        # the library rounds its product at other places: half a bf16 step on either side
        assert rel_l2(got.double().cpu().numpy(), want.double().cpu().numpy()) <= 2 ** -8
        buf = layer._w_buf  # (whose memory would be room)
        layer._set_shared_buf(None)
        with pytest.raises(torch.OutOfMemoryError):
            layer(x)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    del buf
    assert torch.equal(layer(x), want)


@pytest.mark.parametrize("in_f,rows", [(1024, 2), (1024, 16), (1004, 5), (1004, 20)])
def test_calls_that_are_not_plain_keep_the_decode(monkeypatch, dev, in_f, rows):
    """Gradients, forward mode, vmap, autocast and other kinds of tensors: a layer with a decode buffer whose rows went
    through decode + F.linear before it had lanes (dense, not (3,5,8); 17 to 32 rows of a large dense layer) still serves them
    that way, and only plain calls from the lanes."""
    from torch.autograd import forward_ad

    from ixrun_amd import engine

    monkeypatch.setattr(engine, "SPLIT_FUSED_MIN_WEIGHTS", 0)
    products = []

    def linear(x, w, bias):  # in fp32: what is asked for here is who multiplies, and what the caller gets back
        products.append(x.shape)
        return torch.nn.functional.linear(x.float(), w.float(), bias).to(torch.float16 if torch.is_autocast_enabled("cuda") else x.dtype)

    monkeypatch.setattr(engine.gemm_tuning, "linear", linear)
    v, scheme, _ = values("real", 64, in_f)
    p = packed_from_int8(v, 64, in_f, level_bits=scheme)
    layer, plain = engine.StreamingLinear(p), engine.StreamingLinear(p, lanes=False)
    for one in (layer, plain):
        one._set_shared_buf(torch.zeros(p["N"], dtype=torch.bfloat16, device=dev))
    x = activations(rows, in_f, seed=5).to(dev)

    with torch.no_grad():
        layer(x.clone().requires_grad_())
    with torch.autocast("cuda", dtype=torch.bfloat16):
        layer(x)
    y = layer(x)
    assert not products and not bool(layer._w_buf.any())

    def gradient(one):
        leaf = x.clone().requires_grad_()
        one(leaf).sum().backward()
        return leaf.grad

    def tangent(one):
        with forward_ad.dual_level():
            return forward_ad.unpack_dual(one(forward_ad.make_dual(x, x.flip(0)))).tangent

    def mapped(one):
        return torch.vmap(one)(torch.stack([x, x.flip(0)]))

    def cast(one):
        with torch.autocast("cuda", dtype=torch.float16):
            return one(x)

    class Named(torch.Tensor):
        pass

    for call in (gradient, tangent, mapped, cast, lambda one: one(x.as_subclass(Named))):
        del products[:]
        got, n = call(layer), len(products)
        want = call(plain)
        assert n and len(products) == 2 * n and type(got) is type(want) and got.dtype == want.dtype and torch.equal(got, want)
    assert rel_l2(y.double().cpu().numpy(), plain(x).double().cpu().numpy()) <= 2 ** -8


def test_one_hot_rows_are_decoded_columns(oracle, dev):
    out_f, in_f = 24, 1100
    p, lanes = lay_out("real", out_f, in_f, dev)
    w = bits_to_bf16(oracle.decode_packed_bf16(p)).reshape(out_f, in_f)
    cols = [0, 31, 511, 512, 639, 1023, 1024, 1099]
    for m in (1, 8):
        for c0 in range(0, len(cols), m):
            x = torch.zeros((m, in_f), dtype=torch.bfloat16)
            for j in range(m):
                x[j, cols[c0 + j]] = 1
            y = product(lanes, x.to(dev), out_f, in_f).cpu()
            for j in range(m):
                assert torch.equal(y[j], w[:, cols[c0 + j]])


def test_layer_rebuilds_its_lanes_with_its_state(dev):
    """The layout is no part of the state dict and follows the packed streams that are loaded."""
    from ixrun_amd.engine import StreamingLinear

    layers = []
    for seed in (1, 2):
        v = int8_mix("only_l1", 64 * 1024, seed=seed)  # equal level counts: streams of equal length
        layers.append(StreamingLinear(packed_from_int8(v, 64, 1024)))
    assert not any("lane" in k for k in layers[0].state_dict())
    x = activations(1, 1024, seed=9).to(dev)
    assert not torch.equal(layers[0](x), layers[1](x))
    layers[0].load_state_dict(layers[1].state_dict())
    assert torch.equal(layers[0](x), layers[1](x))


def test_state_that_does_not_fit_is_not_followed(monkeypatch, dev):
    """A state of other stream lengths raises, one that holds a part of the streams is loaded: neither has its tables and
    streams decoded together.  The layer goes on with the layout it has, and takes a whole state afterwards."""
    from ixrun_amd.engine import StreamingLinear

    p = [packed_from_int8(int8_mix(kind, 64 * 1000, seed=seed), 64, 1000)
         for kind, seed in (("only_l1", 1), ("no_l3", 2), ("only_l1", 3))]
    layer, longer, other = (StreamingLinear(q) for q in p)
    x = activations(3, 1000, seed=9).to(dev)
    want = layer(x)
    followed = []
    real = StreamingLinear._follow_streams
    monkeypatch.setattr(StreamingLinear, "_follow_streams", lambda self: (followed.append(self), real(self)))
    with pytest.raises(RuntimeError, match="size mismatch"):
        layer.load_state_dict(longer.state_dict())
    state = {k: t.clone() for k, t in other.state_dict().items()}
    layer.load_state_dict({k: state[k] for k in ("_b1", "_scale")}, strict=False)
    layer.load_state_dict({}, strict=False)
    assert not followed and torch.equal(layer(x), want)
    layer.load_state_dict(state)
    assert followed == [layer] and torch.equal(layer(x), other(x))


@pytest.mark.parametrize("in_f", [1024, 1000])
@pytest.mark.parametrize("way", ["moved", "assigned", "assigned on the host"])
def test_layer_follows_a_state_loaded_elsewhere(dev, in_f, way):
    """A state loaded while the layer is on the host, or taken over tensor by tensor: lanes, tables and decode are of the
    new weights once the layer is on the GPU."""
    from ixrun_amd.engine import StreamingLinear

    p = [packed_from_int8(int8_mix("only_l1", 64 * in_f, seed=seed), 64, in_f) for seed in (1, 2)]
    layer, other = StreamingLinear(p[0]), StreamingLinear(p[1])
    if way == "moved":
        layer.cpu()
        layer.load_state_dict(other.state_dict())
        layer.cuda()
    else:
        state = {k: t.to("cpu" if "host" in way else dev, copy=True) for k, t in other.state_dict().items()}
        layer.load_state_dict(state, assign=True)
        del state
        layer.cuda()
    junk = [torch.full((1 << 14,), 3, dtype=torch.int32, device=dev) for _ in range(8)]
    buf = torch.empty(64 * in_f, dtype=torch.bfloat16, device=dev)
    for one in (layer, other):
        one._set_shared_buf(buf)
    assert torch.equal(layer._decode().clone(), other._decode())
    for m in (1, 3, 12):
        x = activations(m, in_f, seed=9).to(dev)
        want = other(x)
        assert torch.equal(layer(x), want)
        layer._lanes, lanes = None, layer._lanes  # and from the packed streams
        layer._native, native, layer._gemv_fn, fn = None, layer._native, lib_gemv(), layer._gemv_fn
        layer._forget_plans()
        assert rel_l2(layer(x).double().cpu().numpy(), want.double().cpu().numpy()) <= 1e-3
        layer._lanes, layer._native, layer._gemv_fn = lanes, native, fn
        layer._forget_plans()
    del junk


def test_layer_without_lanes_stays_without_when_it_loads_a_state(dev):
    from ixrun_amd.engine import StreamingLinear

    p = [packed_from_int8(int8_mix("only_l1", 64 * 1024, seed=seed), 64, 1024) for seed in (1, 2)]
    without, other = StreamingLinear(p[0], lanes=False), StreamingLinear(p[1])
    without.load_state_dict(other.state_dict())
    assert without._lanes is None and not any("lane" in name for name, b in without.named_buffers() if b is not None)
    x = activations(3, 1024, seed=9).to(dev)
    assert rel_l2(without(x).double().cpu().numpy(), other(x).double().cpu().numpy()) <= 1e-3
    other.load_state_dict(without.state_dict())
    assert other._lanes is not None


@pytest.mark.parametrize("in_f", [1024, 1000])
@pytest.mark.parametrize("grows", [False, True])
def test_graph_serves_the_state_that_is_loaded(dev, in_f, grows):
    """A graph captured before load_state_dict: the layer's layout and tables are refreshed in place, and the replay gives the
    new weights' products.  A list that has outgrown its memory takes a new layout, and the old one stays whole: the graph
    gives the old products, and one captured again the new ones."""
    from ixrun_amd.engine import StreamingLinear

    out_f, names = 256, ("_lane_plane", "_lane_off", "_lane_pos", "_lane_val")
    v = [int8_mix("only_l1", out_f * in_f, seed=seed).reshape(out_f, in_f) for seed in (1, 2)]
    for i in range(256):  # as many listed elements: one a row (64 quads), or all in one row and cell (256)
        v[0][i, 5] = 50
        v[1][(0, i) if grows else (i, 7)] = 60
    p = [packed_from_int8(w.reshape(-1), out_f, in_f) for w in v]
    assert p[0]["counts"] == p[1]["counts"]
    layer, other = StreamingLinear(p[0]), StreamingLinear(p[1])
    assert (other._lanes.struct.n_quads > layer._lanes.struct.n_quads) == grows
    xs = [activations(m, in_f, seed=9).to(dev) for m in (1, 8)]
    old, new = [layer(x) for x in xs], [other(x) for x in xs]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ys = [layer(x) for x in xs]
    kept = [weakref.ref(getattr(layer, n)) for n in names]
    sizes = [t().shape for t in kept]
    layer.load_state_dict(other.state_dict())
    for _ in range(3):
        junk = [torch.full(n, 3, dtype=t.dtype, device=dev) for n, t in zip(sizes, layer._lanes.tensors)]  # what freed buffers would be given to
        graph.replay()
        torch.cuda.synchronize()
        for y, want in zip(ys, old if grows else new):
            assert torch.equal(y, want)
        del junk
    for x, want in zip(xs, new):
        assert torch.equal(layer(x), want)
    assert [getattr(layer, n) is t() for n, t in zip(names, kept)] == [not grows] * 4
    assert all(t() is not None for t in kept)
    buf = torch.empty(out_f * in_f, dtype=torch.bfloat16, device=dev)
    for one in (layer, other):
        one._set_shared_buf(buf)
    assert torch.equal(layer._decode().clone(), other._decode())


@pytest.mark.parametrize("kind", ["rare", "real"])
@pytest.mark.parametrize("out_f,in_f,lanes", [(512, 64, False), (3, 700, True), (1, 1000, False), (256, 520, True), (300, 320, True)])
def test_layout_is_not_larger_than_the_weight(oracle, dev, kind, out_f, in_f, lanes):
    """The layout's padding (whole blocks of 4 rows x 512 columns) is bounded: where it would take more than the bf16
    weight, the layer is served from the packed streams."""
    from ixrun_amd.engine import StreamingLinear

    v, scheme, _ = values(kind, out_f, in_f)
    p = packed_from_int8(v, out_f, in_f, level_bits=scheme)
    layer = StreamingLinear(p)
    assert (layer._lanes is not None) == lanes
    if lanes:
        assert layer._lanes.nbytes <= 2 * p["N"] + 4096  # (a list holds 64 quads at least)
    layer._set_shared_buf(torch.empty(p["N"], dtype=torch.bfloat16, device=dev))
    for m in (1, 4, 16, 40):
        x = activations(m, in_f, seed=m)
        check(oracle, p, x, layer(x.to(dev)))


def test_layer_goes_without_lanes_where_memory_is_short(monkeypatch, oracle, dev):
    """A layout that would leave less than a quarter of the GPU's memory is not made; the layer serves from the packed streams."""
    from ixrun_amd.engine import StreamingLinear

    v, scheme, _ = values("real", 64, 1024)
    p = packed_from_int8(v, 64, 1024, level_bits=scheme)
    for free, lanes in ((60, False), (1000, True)):
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (free << 20, 240 << 20))
        layer = StreamingLinear(p)
        assert (layer._lanes is not None) == lanes
        for m in (1, 3, 16):
            x = activations(m, 1024, seed=m)
            check(oracle, p, x, layer(x.to(dev)))


def test_malformed_lanes_are_refused(dev):
    from ixrun_amd import _lib

    L = _lib.lib()
    p, lanes = lay_out("rare", 8, 512, dev)
    x, y = activations(1, 512).to(dev), torch.empty((1, 8), dtype=torch.bfloat16, device=dev)
    call = lambda s, m=1: L.ixh_lanes_gemv(C.byref(s), x.data_ptr(), 512, None, m, y.data_ptr(), 8, None, 0, None)
    for field, value in (("bits", 6), ("plane_words", 100), ("n_quads", 0), ("n_quads", 100), ("n_quads", 1 << 30), ("exc_off", None), ("scale", None)):
        s = _lib.IxhLanes.from_buffer_copy(lanes.struct)
        setattr(s, field, value)
        assert call(s) == -1, field
    assert call(lanes.struct, 0) == -1 and call(lanes.struct, 17) == -1
    many = lambda x, ldx, m, ws=0: L.ixh_lanes_gemm(C.byref(lanes.struct), x, ldx, None, m, y.data_ptr(), 8, None, ws, None)
    assert many(x.data_ptr(), 512, 0) == -1 and many(x.data_ptr(), 512, 4097) == -1 and many(None, 512, 1) == -1
    with pytest.raises(_lib.IxhError, match="16-byte"):
        _lib.check(many(x.data_ptr() + 2, 512, 1))
    assert many(x.data_ptr(), 516, 17) == _lib.IXH_EUNSUPPORTED
    assert L.ixh_lanes_plane_words(8, 512, 7) == -1 and L.ixh_lanes_cells(0, 512) == -1


@pytest.mark.parametrize("out_f,in_f", [(7, 1000), (33, 513), (5, 4099)])
def test_rows_of_other_lengths_decode_by_flat_units(oracle, dev, out_f, in_f):
    """A layer whose rows are not whole units of 512 decodes by units counted over the row ends, also after another
    layer's state has been loaded into it."""
    from ixrun_amd.engine import StreamingLinear

    v, scheme, _ = values("real", out_f, in_f)
    packed = [packed_from_int8(w, out_f, in_f, level_bits=scheme) for w in (v, np.roll(v, 3))]
    want = [oracle.decode_packed_bf16(p).reshape(-1) for p in packed]
    layers = [StreamingLinear(p) for p in packed]
    for layer, w in zip(layers, want):
        layer._set_shared_buf(torch.empty(out_f * in_f, dtype=torch.bfloat16, device=dev))
        assert np.array_equal(bf16_bits(layer._decode()).reshape(-1), w)
    layers[0].load_state_dict(layers[1].state_dict())
    assert np.array_equal(bf16_bits(layers[0]._decode()).reshape(-1), want[1])


def test_forward_in_native_code_takes_only_the_common_case(oracle, dev):
    """Contiguous bf16 activations of 1 to 16 rows go through the native forward, with any leading dimensions; the rest
    (views, other row lengths, other types, 17 rows) is left to the code behind it, which has to give the same."""
    from ixrun_amd.engine import StreamingLinear

    v, scheme, _ = values("real", 24, 1024)
    p = packed_from_int8(v, 24, 1024, level_bits=scheme)
    bias = torch.randn(24, generator=torch.Generator().manual_seed(1)).bfloat16()
    layer = StreamingLinear(p, bias=bias)
    layer._set_shared_buf(torch.empty(p["N"], dtype=torch.bfloat16, device=dev))
    x = activations(16, 1024, seed=4).to(dev)
    want = layer(x)
    assert torch.equal(layer._native(x), want)
    assert torch.equal(layer(x.view(2, 8, 1024)), want.view(2, 8, 24)) and torch.equal(layer(x[3]), layer(x[3:4])[0])
    for other in (x.t().contiguous().t(), torch.cat([x, x])[::2], x[:, :512], x.float(), x.cpu(), torch.cat([x, x[:1]]), x[:0]):
        assert layer._native(other) is None
    assert torch.equal(layer(x.t().contiguous().t()), want)
    assert layer(x[:0]).shape == (0, 24)
    with pytest.raises(TypeError):
        layer._native.__init__(1, 2)
