"""Parity of the gfx950 kernels with the CPU oracle, through the C ABI.

Integer results (rank tables, decoded int8, decoded bf16 bit patterns) must be
bit-exact.  Fused decode+GEMV outputs are compared with the fp64 oracle on the
same seeded inputs: relative L2 error <= 1e-3 (the build's tolerance) and the
reference's own acceptance metric max|dy| / max|y| < 5e-3
(tests/test_fused.py:34-37, tests/test_splitk.py:34-35).
"""
import numpy as np
import pytest
import torch

from helpers import (activations, bf16_bits, calibrated_weight, int8_mix, outlier_weight, packed_from_int8, rel_l2,
                     student_t_weight)

pytestmark = pytest.mark.gpu

REL_L2_TOL = 1e-3
REF_MAX_TOL = 5e-3


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from ixrun_amd import _lib

    assert _lib.lib().ixh_version() >= 100  # the HIP library itself, not a fallback
    return torch.device("cuda:0")


def quantize(w, level_bits=(3, 5, 8)):
    from ixrun_amd.quantize import int8x_quantize

    return int8x_quantize(w, level_bits)


def device_packed(p, dev):
    from ixrun_amd import _lib

    return _lib.DevicePacked.from_dict(p, dev)


def check_outputs(y, y64, what=""):
    """y: bf16 bit patterns (uint16) or fp32 values, against the fp64 oracle.

    fp32 results (partial sums before the output rounding) must agree with the
    fp64 oracle to 2e-5 relative L2: only the order of the fp32 additions
    separates them.  bf16 results are compared with the oracle rounded to bf16,
    the output type, as the reference's own check compares two bf16 vectors:
    relative L2 <= 1e-3, and the reference's criterion max|dy| / max|y| < 5e-3.
    (Against the unrounded fp64 value any bf16 vector sits near 1.6e-3, the
    rounding noise of an 8-bit significand.)
    """
    if y.dtype == np.float32:
        err = rel_l2(y, y64)
        assert err <= 2e-5, f"{what}: fp32 rel-L2 {err:.3e}"
        return err
    from oracle import ix_oracle

    yv = ix_oracle.bf16_bits_to_f32(y).astype(np.float64).reshape(y64.shape)
    want = ix_oracle.bf16_bits_to_f32(ix_oracle.f32_to_bf16_bits(y64.astype(np.float32))).astype(np.float64)
    err = rel_l2(yv, want)
    ref_metric = np.abs(yv - y64).max() / max(np.abs(y64).max(), 1e-300)
    assert err <= REL_L2_TOL, f"{what}: rel-L2 {err:.3e}"
    assert ref_metric < REF_MAX_TOL, f"{what}: max-rel {ref_metric:.3e}"
    return err


def make_packed(kind, out_f, in_f, level_bits=(3, 5, 8)):
    """Packed dictionaries with the level mixes the kernels must survive."""
    if kind == "outlier":
        return quantize(outlier_weight(out_f, in_f, seed=0), level_bits)
    if kind == "student_t":
        return quantize(student_t_weight(out_f, in_f, seed=0), level_bits)
    if kind == "calibrated_pow2":
        return quantize(calibrated_weight(out_f, in_f, seed=0)[0], level_bits)
    if kind == "calibrated_odd_scale":  # scale bf16(0.0123): v*scale is rounded when dequantised
        return quantize(calibrated_weight(out_f, in_f, seed=0, scale=0.0123046875)[0], level_bits)
    return packed_from_int8(int8_mix(kind, out_f * in_f, seed=1), out_f, in_f, level_bits=level_bits)


KINDS = ["outlier", "student_t", "calibrated_pow2", "calibrated_odd_scale", "only_l1", "no_l3", "no_l2", "only_l3",
         "rare_other"]


# ---------------------------------------------------------------- rank tables
@pytest.mark.parametrize("shape,level_bits,chunk", [
    ((64, 1024), (3, 5, 8), 512), ((96, 1024), (3, 5, 8), 1024), ((33, 96), (3, 4, 5, 6, 8), 32),
    ((5, 7), (3, 5, 8), 7), ((17, 100), (3, 5, 8), 1024), ((300, 1536), (3, 5, 8), 512), ((7, 33), (2, 8), 5),
    # more table entries than one scan tile of 8192: 38 664, 73 728 (nine whole tiles) and 8193 units
    ((300, 1031), (3, 5, 8), 8), ((256, 4608), (3, 4, 5, 6, 8), 16), ((8193, 4), (3, 5, 8), 4), ((2048, 2048), (3, 5, 8), 512)])
def test_prefix_build(oracle, dev, shape, level_bits, chunk):
    p = quantize(outlier_weight(*shape, seed=7), level_bits)
    dp = device_packed(p, dev)
    table = dp.prefix_build(chunk).cpu().numpy()
    pn = oracle.packed_to_numpy(p)
    want = oracle.prefix(p["N"], len(level_bits), pn["bitmaps"], chunk)
    assert table.shape == want.shape and np.array_equal(table, want)


def test_reference_shaped_tables(oracle, dev):
    from ixrun_amd.fused import compute_row_prefixes
    from ixrun_amd.triton_kernels import precompute_block_offsets

    p = quantize(outlier_weight(48, 2048, seed=3))
    b1_blk, b2_blk = precompute_block_offsets(p, device=dev)
    pn = oracle.packed_to_numpy(p)
    want = oracle.prefix(p["N"], 3, pn["bitmaps"], 1024)
    assert b1_blk.dtype == torch.int32 and b1_blk.is_cuda and b1_blk.numel() == p["N"] // 1024
    assert np.array_equal(b1_blk.cpu().numpy(), want[0, :-1]) and np.array_equal(b2_blk.cpu().numpy(), want[1, :-1])
    q1, q2 = compute_row_prefixes(p, 1024)
    assert np.array_equal(q1.numpy(), want[0, :-1]) and np.array_equal(q2.numpy(), want[1, :-1])


# ---------------------------------------------------------------- decode, bit-exact
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(1, 1), (3, 11), (7, 33), (128, 256), (33, 1000), (64, 1536), (300, 1031)])
def test_decode_bit_exact(oracle, dev, kind, shape):
    p = make_packed(kind, *shape)
    dp = device_packed(p, dev)
    q_want = oracle.decode_packed_i8(p)
    w_want = oracle.decode_packed_bf16(p)
    for chunk in (1024, 512, 96):
        table = dp.prefix_build(chunk)
        o8 = torch.full((p["N"],), 99, dtype=torch.int8, device=dev)
        o16 = torch.zeros(p["N"], dtype=torch.bfloat16, device=dev)
        dp.decode(table, chunk, out_i8=o8, out_bf16=o16)
        assert np.array_equal(o8.cpu().numpy(), q_want), (kind, shape, chunk)
        assert np.array_equal(bf16_bits(o16).reshape(shape), w_want), (kind, shape, chunk)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(1, 512), (3, 171), (33, 1000), (64, 1536), (300, 1031), (256, 4608)])
@pytest.mark.parametrize("level_bits", [(3, 5, 8), (3, 4, 5, 6, 8), (2, 8), (5, 6, 7, 8)])
def test_decode_bf16_only(oracle, dev, kind, shape, level_bits):
    """bf16-only decode at the 512-element table unit: the kernel that stages the streams in LDS
    (ragged last unit, rows that are not whole units, level-1 codes wider than 4 bits)."""
    p = make_packed(kind, *shape, level_bits)
    dp = device_packed(p, dev)
    table = dp.prefix_build(512)
    o16 = torch.full((p["N"] + 8,), 7.0, dtype=torch.bfloat16, device=dev)
    dp.decode(table, 512, out_bf16=o16[: p["N"]])
    assert np.array_equal(bf16_bits(o16[: p["N"]]).reshape(shape), oracle.decode_packed_bf16(p)), (kind, shape, level_bits)
    assert torch.all(o16[p["N"]:] == 7.0)  # nothing written past the end


@pytest.mark.parametrize("decoder", ["staged", "dense", "rows"])
@pytest.mark.parametrize("kind", KINDS + ["all_l3", "zeros"])
@pytest.mark.parametrize("shape", [(1, 1), (1, 31), (1, 512), (3, 171), (5, 413), (33, 1000), (64, 1536), (300, 1031),
                                   (256, 4608), (17, 2048), (1, 2049), (4, 512), (8, 512), (52, 512), (200, 1024),
                                   (1000, 2048), (2600, 1024)])
def test_decode_358_each_decoder(oracle, dev, force_decoder, kind, shape, decoder):
    """(3,5,8) to bf16 at unit 512 through each of the three decoders, whatever the mix of levels would choose:
    the level-by-level one (partial last lane, partial last span, tensors smaller than a lane), the one that
    stages the streams, and the row-block one (whole unit-quads only: other sizes fall through to the staged one;
    with dense mixes its record queue is resolved every few units)."""
    force_decoder(decoder)
    if kind == "all_l3":
        g = torch.Generator("cpu").manual_seed(shape[1])
        w = ((torch.randint(0, 2, shape, generator=g) * 2 - 1) * (0.25 + 0.5 * torch.rand(shape, generator=g))).bfloat16()
        p = quantize(w, (3, 5, 8))
    elif kind == "zeros":
        p = quantize(torch.zeros(shape, dtype=torch.bfloat16), (3, 5, 8))
    else:
        p = make_packed(kind, *shape, (3, 5, 8))
    dp = device_packed(p, dev)
    table = dp.prefix_build(512)
    o16 = torch.full((p["N"] + 64,), 7.0, dtype=torch.bfloat16, device=dev)
    dp.decode(table, 512, out_bf16=o16[: p["N"]])
    assert np.array_equal(bf16_bits(o16[: p["N"]]).reshape(shape), oracle.decode_packed_bf16(p)), (kind, shape, decoder)
    assert torch.all(o16[p["N"]:] == 7.0)  # nothing written past the end


@pytest.mark.parametrize("decoder", ["auto", "dense"])
@pytest.mark.parametrize("kind", KINDS + ["five_dense", "zeros"])
@pytest.mark.parametrize("shape", [(1, 1), (1, 31), (1, 512), (3, 171), (5, 413), (33, 1000), (64, 1536), (300, 1031),
                                   (256, 4608), (17, 2048), (1, 2049), (52, 512), (1000, 2048)])
def test_decode_34568_level_by_level(oracle, dev, force_decoder, kind, shape, decoder):
    """(3,4,5,6,8) to bf16 at unit 512 through the five-level level-by-level decoder: what the library picks for dense
    mixes, forced for the others (partial last lane, partial last span, tensors smaller than a lane)."""
    force_decoder(decoder)
    if kind == "zeros":
        p = quantize(torch.zeros(shape, dtype=torch.bfloat16), (3, 4, 5, 6, 8))
    else:
        p = make_packed(kind, *shape, (3, 4, 5, 6, 8))
    dp = device_packed(p, dev)
    table = dp.prefix_build(512)
    o16 = torch.full((p["N"] + 64,), 7.0, dtype=torch.bfloat16, device=dev)
    dp.decode(table, 512, out_bf16=o16[: p["N"]])
    assert np.array_equal(bf16_bits(o16[: p["N"]]).reshape(shape), oracle.decode_packed_bf16(p)), (kind, shape, decoder)
    assert torch.all(o16[p["N"]:] == 7.0)  # nothing written past the end


@pytest.mark.parametrize("level_bits", [(3, 4, 5, 6, 8), (3, 8), (3, 3, 8), (3, 4, 8), (3, 5, 6, 7, 8), (3, 4, 5, 6, 7, 8)])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(8, 512), (64, 1536), (1000, 2048)])
def test_decode_row_block_decoder_other_schemes(oracle, dev, force_decoder, kind, shape, level_bits):
    """The row-block decoder takes every scheme whose first level has 3 bits; its elements above level 1 are followed
    down the nested bitmaps one by one.  Forced here for every mix (it is chosen only for tensors that are almost all
    level 1)."""
    force_decoder("rows")
    p = make_packed(kind, *shape, level_bits)
    dp = device_packed(p, dev)
    table = dp.prefix_build(512)
    o16 = torch.full((p["N"] + 64,), 7.0, dtype=torch.bfloat16, device=dev)
    dp.decode(table, 512, out_bf16=o16[: p["N"]])
    assert np.array_equal(bf16_bits(o16[: p["N"]]).reshape(shape), oracle.decode_packed_bf16(p)), (kind, shape, level_bits)
    assert torch.all(o16[p["N"]:] == 7.0)


@pytest.mark.parametrize("level_bits", [(3, 4, 5, 6, 8), (2, 8), (4, 8), (1, 2, 3, 4, 5, 6, 7, 8), (3, 3, 8)])
def test_decode_other_level_schemes(oracle, dev, level_bits):
    from ixrun_amd.triton_kernels import decode_weight_triton, decode_int8

    p = quantize(outlier_weight(96, 200, seed=9), level_bits)
    assert np.array_equal(decode_int8(p, dev).cpu().numpy().reshape(-1), oracle.decode_packed_i8(p))
    w = decode_weight_triton(p, device=dev)
    assert w.dtype == torch.bfloat16 and w.shape == (96, 200)
    assert np.array_equal(bf16_bits(w), oracle.decode_packed_bf16(p))


def test_decode_config1_2048(oracle, dev):
    """2048x2048 Student-t, int8 round trip bit-exact, level fractions reported."""
    from ixrun_amd.triton_kernels import decode_weight_triton, decode_int8

    w = student_t_weight(2048, 2048, seed=0)
    p = quantize(w)
    scale_bits, q = oracle.quantize_bf16(bf16_bits(w))
    assert np.array_equal(decode_int8(p, dev).cpu().numpy().reshape(-1), q)
    assert np.array_equal(bf16_bits(decode_weight_triton(p, device=dev)).reshape(-1), oracle.dequant_bf16(q, scale_bits))
    frac = [c / p["N"] for c in p["counts"]]
    print(f"config1 fractions L1/L2/L3 = {frac[0]:.4f}/{frac[1]:.4f}/{frac[2]:.5f}, bpw {p['bits_per_weight']:.3f}")
    assert p["total_bytes"] == 2_336_569  # byte accounting of this seeded recipe: a change in the generator or the encoder shows up here


# ---------------------------------------------------------------- fused decode + GEMV
def test_gemv_config1_2048(oracle, dev):
    """The fused path: ixh_gemv on the 2048 x 2048 Student-t tensor, one activation row,
    against the fp64 oracle; once with the kernel the library picks for this mix, once with the (3,5,8) row-block
    kernels forced (IXH_GEMV_FORCE_358), bf16 output and the fp32 atomic mode."""
    from ixrun_amd import _lib

    p = quantize(student_t_weight(2048, 2048, seed=0))
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    x = activations(1, 2048, seed=0)
    y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
    for flags in (0, _lib.IXH_GEMV_FORCE_358):
        for atomic in (False, True):
            y = run_gemv(dp, 512, x, 1, dev, flags=flags, atomic=atomic)
            check_outputs(y, y64, f"config 1 flags={flags} atomic={atomic}")


def test_gemv_binding_rejects_bad_buffers(dev):
    """The Python binding checks every buffer of a fused call before the library sees a pointer: outputs on the host,
    of the wrong type, too small or strided, a rank table for another chunk, a workspace on the host."""
    p = quantize(outlier_weight(8, 1024, seed=1))
    dp = device_packed(p, dev)
    table = dp.prefix_build(512)
    x = activations(2, 1024, seed=1).to(dev)
    ok = torch.zeros((2, 8), dtype=torch.bfloat16, device=dev)
    ws = torch.empty(dp.gemv_workspace_bytes(512, 2) // 4, dtype=torch.float32, device=dev)
    dp.gemv(table, 512, x, y=ok, workspace=ws)
    wide = torch.zeros((2, 16), dtype=torch.bfloat16, device=dev)
    dp.gemv(table, 512, x, y=wide[:, :8], workspace=ws)  # rows 16 elements apart: ldy
    torch.cuda.synchronize()
    assert torch.equal(wide[:, :8], ok) and torch.all(wide[:, 8:] == 0)
    bad = [
        dict(y=ok.cpu()), dict(y=ok.float()), dict(y=ok[:1]), dict(y=torch.zeros((2, 4), dtype=torch.bfloat16, device=dev)),
        dict(y=wide.t()[:8].t()[:, ::2]), dict(y=None, y32=torch.zeros((2, 8), dtype=torch.bfloat16, device=dev)),
        dict(y=None, y32=torch.zeros(15, dtype=torch.float32, device=dev)),
        dict(y=ok, table=dp.prefix_build(256)), dict(y=ok, table=table.cpu()), dict(y=ok, table=table.long()),
        dict(y=ok, workspace=ws.cpu()), dict(y=ok, workspace=torch.empty((4, 64), device=dev)[:, ::2]),
    ]
    for kw in bad:
        args = dict(table=table, y32=None, workspace=ws)
        args.update(kw)
        with pytest.raises((ValueError, RuntimeError)) as e:
            dp.gemv(args["table"], 512, x, y=args["y"], y32=args["y32"], workspace=args["workspace"])
        assert not isinstance(e.value, _lib_error())
    with pytest.raises((ValueError, RuntimeError)):
        dp.gemv_noalloc(table, 512, x, ok.float())
    with pytest.raises(ValueError):
        dp.gemv_noalloc(table, 512, x, None)


def _lib_error():
    from ixrun_amd import _lib

    return _lib.IxhError


def run_gemv(dp, chunk, x, m, dev, flags=0, atomic=False):
    from ixrun_amd import _lib

    table = dp.prefix_build(chunk)
    xd = x.to(dev)
    if atomic:
        y32 = torch.zeros((m, dp.out_f), dtype=torch.float32, device=dev)
        dp.gemv(table, chunk, xd, y32=y32, flags=flags | _lib.IXH_GEMV_ATOMIC)
        return y32.cpu().numpy()
    y = torch.zeros((m, dp.out_f), dtype=torch.bfloat16, device=dev)
    nbytes = dp.gemv_workspace_bytes(chunk, m, flags)
    ws = torch.empty(max(nbytes // 4, 1), dtype=torch.float32, device=dev)
    dp.gemv(table, chunk, xd, y=y, workspace=ws, flags=flags)
    return bf16_bits(y)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(64, 512), (37, 1024), (130, 1536), (256, 4608)])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 7, 8, 9, 13, 16])
def test_gemv_fast_and_general(oracle, dev, kind, shape, m):
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f)
    dp = device_packed(p, dev)
    x = activations(m, in_f, seed=1)
    y64 = oracle.gemm_f64(oracle.decode_packed_bf16(p), bf16_bits(x))
    for flags, chunk, atomic in [(0, 512, False), (_lib.IXH_GEMV_FORCE_358, 512, False), (0, 512, True),
                                 (_lib.IXH_GEMV_FORCE_358, 512, True), (_lib.IXH_GEMV_COLUMN_KERNEL, 512, False),
                                 (_lib.IXH_GEMV_FORCE_GENERIC, 512, False),
                                 (0, in_f, False), (0, 256, True)]:
        y = run_gemv(dp, chunk, x, m, dev, flags=flags, atomic=atomic)
        check_outputs(y, y64, f"{kind} {shape} m={m} flags={flags} chunk={chunk} atomic={atomic}")
    if m <= 8:  # the level-by-level kernels (one row; 2..8 rows), forced also for the mixes they are not built for
        for atomic in (False, True):
            y = run_gemv(dp, 512, x, m, dev, flags=_lib.IXH_GEMV_DENSE, atomic=atomic)
            check_outputs(y, y64, f"{kind} {shape} m={m} level-by-level kernel atomic={atomic}")


@pytest.mark.parametrize("kind", KINDS + ["five_dense"])
@pytest.mark.parametrize("shape", [(64, 1024), (37, 1024), (130, 1536), (256, 4608), (24, 8704), (21, 17408), (5, 25600), (300, 2048)])
@pytest.mark.parametrize("cus", [0, 1, 3, 7])
@pytest.mark.parametrize("level_bits", [(3, 5, 8), (3, 4, 5, 6, 8)])
def test_gemv_dense_rows_on_the_matrix_pipe(oracle, dev, gemv_option, kind, shape, cus, level_bits):
    """The level-by-level kernel for 2..16 activation rows that multiplies 16 rows' spans on the matrix pipe, forced
    for every mix: row counts that are not multiples of 16 (waves without a row), rows whose last span is short,
    the steps dealt to 1, 3, 7 or all workgroups, so that workgroups hold several row blocks and row blocks lie in
    several workgroups (pieces added by the second kernel); the (3,5,8) kernel and the five-level one (the full
    decoder in its tile mode); and the (3,5,8) kernel it replaced for 2..8 rows, still reachable."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f, level_bits)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    gemv_option("gemv_tile_cus", cus)
    for m in (2, 3, 8, 9, 16):
        x = activations(m, in_f, seed=m)
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        for dense_tiles in (1, 0, -1) if (m <= 8 and cus == 0 and len(level_bits) == 3) else (1,):
            gemv_option("gemv_dense_tiles", dense_tiles)
            y = run_gemv(dp, 512, x, m, dev, flags=_lib.IXH_GEMV_DENSE)
            check_outputs(y, y64, f"{kind} {shape} m={m} on {cus} CUs, gemv_dense_tiles={dense_tiles}")


@pytest.mark.parametrize("kind", ["student_t", "calibrated_odd_scale", "rare_other", "only_l3"])
@pytest.mark.parametrize("shape", [(24, 8704), (21, 17408), (9, 25600), (70, 5120)])
def test_gemv_wide_rows(oracle, dev, kind, shape):
    """Wide rows: 10 to 50 column blocks, so that waves of the row-block kernel own 1 to 4 blocks
    and workgroups end on ragged row quads."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    for m in (1, 2, 4, 7):
        x = activations(m, in_f, seed=m)
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        for flags in (0, _lib.IXH_GEMV_FORCE_358, _lib.IXH_GEMV_COLUMN_KERNEL) + ((_lib.IXH_GEMV_DENSE,) if m <= 8 else ()):
            check_outputs(run_gemv(dp, 512, x, m, dev, flags=flags), y64, f"{kind} {shape} m={m} flags={flags}")


@pytest.mark.parametrize("kind", ["student_t", "rare_other", "only_l1"])
@pytest.mark.parametrize("shape", [(8, 25600), (12, 33792), (4, 57344), (40, 5120), (4, 512)])
def test_gemv_shared_x_kernel_lds_limits(oracle, dev, kind, shape):
    """The row-block kernel that keeps the activation rows in LDS, at the edges of what LDS holds: whole row quads
    with 50, 66 and 112 column blocks (12 waves, 8 waves, and no fit at all: the next kernel takes over), eight
    activation rows beside 10 and 50 column blocks (fit / no fit), waves without a unit-quad of their own."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    for m in (1, 2, 3, 4, 6, 8, 16):
        x = activations(m, in_f, seed=10 + m)
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        for flags in (0, _lib.IXH_GEMV_FORCE_358):
            check_outputs(run_gemv(dp, 512, x, m, dev, flags=flags), y64, f"{kind} {shape} m={m} flags={flags}")


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(8, 512), (64, 512), (40, 1536), (20, 17408), (68, 5120), (256, 4608), (1024, 2048), (4, 33792)])
@pytest.mark.parametrize("level_bits", [(3, 5, 8), (3, 4, 5, 6, 8)])
@pytest.mark.parametrize("kernel", ["strips", "tiles"])
def test_gemv_strip_and_tile_kernels(oracle, dev, gemv_option, kind, shape, level_bits, kernel):
    """The two kernels that take their products on the matrix pipe, each forced for every mix and every number of
    activation rows (by themselves the strip kernel takes 3..8 rows, the tile kernel 9..16 where a workgroup's rows
    fill its 16-row tiles): 1..16 rows, bf16 output and the fp32 accumulate contract, one and several tasks per worker,
    workgroups with fewer tasks than workers, tiles with fewer than 16 rows, activations held in LDS one part of the
    columns at a time (tile kernel, wide rows), dense mixes that overflow the record queues and the shared task list."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f, level_bits)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    gemv_option("gemv_strips", 1)
    gemv_option("gemv_tiles", 1 if kernel == "tiles" else -1)
    for m in (1, 2, 3, 4, 5, 8, 11, 16):
        x = activations(m, in_f, seed=m)
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        for atomic in (False, True):
            y = run_gemv(dp, 512, x, m, dev, flags=_lib.IXH_GEMV_FORCE_358, atomic=atomic)
            check_outputs(y, y64, f"{kernel} {kind} {shape} {level_bits} m={m} atomic={atomic}")


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(8, 512), (64, 512), (40, 1536), (20, 17408), (68, 5120), (256, 4608), (1024, 2048), (12, 33792),
                                   (4, 57344)])
@pytest.mark.parametrize("level_bits", [(3, 5, 8), (3, 4, 5, 6, 8)])
@pytest.mark.parametrize("waves", [0, 8, 13])
def test_gemv_slot_kernel(oracle, dev, gemv_option, kind, shape, level_bits, waves):
    """The row-block decode with its products on the matrix pipe (16 (row, column block) pairs per instruction),
    forced for every mix at one to four activation rows, bf16 output and the fp32 accumulate contract: waves with
    one, several and no groups of their own, a last group with unit-quads past the end, workgroups of 8, 13 and the
    planner's number of waves, dense mixes that fill the record queue inside every group (and the resolver that
    reads global memory), 66 column blocks beside the per-wave stages, 112 column blocks (no fit: the next kernel)."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f, level_bits)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    gemv_option("gemv_slots", 1)
    gemv_option("gemv_slot_waves", waves)
    gemv_option("gemv_tiles", -1)
    gemv_option("gemv_strips", -1)
    for m in (1, 2, 3, 4):
        x = activations(m, in_f, seed=20 + m)
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        for atomic in (False, True):
            y = run_gemv(dp, 512, x, m, dev, flags=_lib.IXH_GEMV_FORCE_358, atomic=atomic)
            check_outputs(y, y64, f"slots {kind} {shape} {level_bits} waves={waves} m={m} atomic={atomic}")


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(20, 512), (36, 1024), (68, 5120), (132, 1536), (100, 8704), (48, 17408)])
@pytest.mark.parametrize("level_bits", [(3, 5, 8), (3, 4, 5, 6, 8)])
@pytest.mark.parametrize("tile_rows", [4, 8, 16])
@pytest.mark.parametrize("cus", [1, 3])
def test_gemv_tile_shapes(oracle, dev, gemv_option, kind, shape, level_bits, tile_rows, cus):
    """The tile kernel with each of its tile shapes forced (4, 8 or 16 weight rows by 4, 2 or 1 column blocks side by
    side; a shape that cannot serve that many activation rows hands the call on to the next kernel), the rows spread
    over one and over three CUs so that a workgroup holds several tiles, a last tile with rows missing, steps whose last
    slots have no column block, activations held in LDS one part of the columns at a time, queues that are emptied
    between tasks (dense mixes), every element above level 1 through the matrix pipe."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f, level_bits)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    gemv_option("gemv_tiles", 1)
    gemv_option("gemv_tile_rows", {4: 2, 8: 3, 16: 4}[tile_rows])
    gemv_option("gemv_tile_cus", cus)
    for m in (1, 2, 3, 4, 5, 8, 11, 16):
        x = activations(m, in_f, seed=m)
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        for atomic in (False, True):
            y = run_gemv(dp, 512, x, m, dev, flags=_lib.IXH_GEMV_FORCE_358, atomic=atomic)
            check_outputs(y, y64, f"tiles of {tile_rows} on {cus} CUs {kind} {shape} {level_bits} m={m} atomic={atomic}")


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(20, 1024), (68, 5120), (132, 1536), (100, 8704), (48, 17408), (132, 512)])
@pytest.mark.parametrize("level_bits", [(3, 5, 8), (3, 4, 5, 6, 8)])
@pytest.mark.parametrize("split", [2, 3, 4, 7])
def test_gemv_tile_split(oracle, dev, gemv_option, kind, shape, level_bits, split):
    """The tile kernel with several workgroups to a block of rows, each taking a run of the rows' column blocks: the
    pieces go through the workspace (filled with NaN before the call: every piece must be written) and a second launch
    that adds them, or one by one into the caller's fp32 sums; row blocks several times as tall, pieces of unequal
    length, pieces held in LDS in several parts, a split that would leave a piece empty (the call then goes on to the
    next kernel), no workspace at all (in_f = 512: a row is one column block, ixh_gemv_workspace_bytes is 0, and the tile
    kernel runs with whole rows per workgroup whatever split is asked for); the same call twice gives the same bits.
    The last call, with chunk = in_f, is served by the wave-per-unit kernel for every in_f but 512 (the other kernels
    take chunk = 512 only) and checks that the options leave it alone."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f, level_bits)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    gemv_option("gemv_tiles", 1)
    gemv_option("gemv_tile_split", split)
    for cus in (2, 8):
        gemv_option("gemv_tile_cus", cus)
        for m in (3, 8, 16):
            x = activations(m, in_f, seed=m)
            y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
            what = f"split {split} on {cus} CUs {kind} {shape} {level_bits} m={m}"
            y = run_gemv(dp, 512, x, m, dev, flags=_lib.IXH_GEMV_FORCE_358, atomic=True)
            check_outputs(y, y64, what + " atomic")
            table = dp.prefix_build(512)
            xd = x.to(dev)
            outs = []
            for _ in range(2):
                yd = torch.zeros((m, out_f), dtype=torch.bfloat16, device=dev)
                nbytes = dp.gemv_workspace_bytes(512, m, _lib.IXH_GEMV_FORCE_358)
                ws = torch.full((max(nbytes // 4, 1),), float("nan"), dtype=torch.float32, device=dev)
                dp.gemv(table, 512, xd, y=yd, workspace=ws, flags=_lib.IXH_GEMV_FORCE_358)
                outs.append(bf16_bits(yd))
            check_outputs(outs[0], y64, what)
            assert np.array_equal(outs[0], outs[1]), what + ": two calls differ"
            y = run_gemv(dp, in_f, x, m, dev, flags=_lib.IXH_GEMV_FORCE_358)
            check_outputs(y, y64, what + " chunk = in_f")


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(64, 512), (37, 1024), (130, 2048), (24, 8704), (5, 25600)])
@pytest.mark.parametrize("level_bits", [(3, 5, 8), (3, 4, 5, 6, 8), (5, 8)])
def test_gemv_staged(oracle, dev, kind, shape, level_bits):
    """The any-scheme kernel that stages the streams in LDS: sparse and dense mixes, rows cut into pieces
    (workspace and atomic combination), level-1 codes wider than 4 bits."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f, level_bits)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    for m in (1, 3, 16):
        x = activations(m, in_f, seed=m)
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        for atomic in (False, True):
            y = run_gemv(dp, 512, x, m, dev, flags=_lib.IXH_GEMV_STAGED, atomic=atomic)
            check_outputs(y, y64, f"{kind} {shape} {level_bits} m={m} atomic={atomic}")


@pytest.mark.parametrize("kind", KINDS + ["five_dense"])
@pytest.mark.parametrize("shape", [(64, 512), (37, 1024), (130, 2048), (300, 1536), (24, 8704), (5, 25600)])
def test_gemv_five_level_dense_kernel(oracle, dev, kind, shape):
    """The level-by-level kernel of the five-level scheme (3,4,5,6,8), one activation row: what the library picks for
    dense mixes, forced for the others; whole rows per wave and spans through the workspace, and the split-K call."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f, (3, 4, 5, 6, 8))
    dp = device_packed(p, dev)
    x = activations(1, in_f, seed=3)
    y64 = oracle.gemm_f64(oracle.decode_packed_bf16(p), bf16_bits(x))
    for flags in (0, _lib.IXH_GEMV_DENSE):
        for atomic in (False, True):
            y = run_gemv(dp, 512, x, 1, dev, flags=flags, atomic=atomic)
            check_outputs(y, y64, f"{kind} {shape} five-level flags={flags} atomic={atomic}")


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(64, 512), (37, 1024), (130, 1536), (24, 8704), (9, 25600)])
@pytest.mark.parametrize("level_bits", [(3, 4, 5, 6, 8), (3, 8), (3, 3, 8), (3, 5, 6, 7, 8)])
def test_gemv_row_block_kernel_other_schemes(oracle, dev, kind, shape, level_bits):
    """The row-block kernel takes every scheme whose first level has 3 bits (its elements above level 1 are followed
    down the nested bitmaps): chosen by itself for tensors that are almost all level 1, forced here for every mix;
    1..4 rows in one launch, 9..16 rows eight (or four) at a time."""
    from ixrun_amd import _lib

    out_f, in_f = shape
    p = make_packed(kind, out_f, in_f, level_bits)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    for m in (1, 2, 4, 9, 16):
        x = activations(m, in_f, seed=m)
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        for flags in (0, _lib.IXH_GEMV_FORCE_358):
            check_outputs(run_gemv(dp, 512, x, m, dev, flags=flags), y64, f"{kind} {shape} {level_bits} m={m} flags={flags}")


@pytest.mark.parametrize("shape,level_bits,chunk", [((40, 96), (3, 4, 5, 6, 8), 32), ((33, 100), (3, 5, 8), 50),
                                                    ((64, 1024), (3, 4, 5, 6, 8), 512), ((9, 7), (2, 8), 7)])
def test_gemv_general_shapes_and_schemes(oracle, dev, shape, level_bits, chunk):
    p = quantize(outlier_weight(*shape, seed=4), level_bits)
    dp = device_packed(p, dev)
    for m in (1, 5):
        x = activations(m, shape[1], seed=2)
        y64 = oracle.gemm_f64(oracle.decode_packed_bf16(p), bf16_bits(x))
        check_outputs(run_gemv(dp, chunk, x, m, dev), y64, f"{shape} {level_bits} m={m}")


@pytest.mark.parametrize("kind", ["student_t", "calibrated_odd_scale", "rare_other"])
def test_gemv_one_hot_is_exact(oracle, dev, kind):
    """x = e_k makes y the decoded column k, exactly: products with 1.0 and zeros add without rounding."""
    out_f, in_f = 96, 1024
    p = make_packed(kind, out_f, in_f)
    dp = device_packed(p, dev)
    w_want = oracle.decode_packed_bf16(p)
    for k in (0, 31, 32, 511, 512, 1023):
        x = torch.zeros(1, in_f, dtype=torch.bfloat16)
        x[0, k] = 1.0
        for chunk in (512, in_f):
            assert np.array_equal(run_gemv(dp, chunk, x, 1, dev)[0], w_want[:, k]), (kind, k, chunk)


@pytest.mark.parametrize("kind", ["student_t", "rare_other"])
@pytest.mark.parametrize("kernel", ["strips", "tiles", "tiles of 8", "tiles of 4"])
def test_gemv_matrix_pipe_kernels_one_hot_is_exact(oracle, dev, gemv_option, kind, kernel):
    """One-hot activation rows through the strip and the tile kernel: every output equals a decoded weight, exactly
    (the matrix pipe multiplies by 1.0 and adds zeros; the elements above level 1 take the same way)."""
    out_f, in_f = 96, 1024
    p = make_packed(kind, out_f, in_f)
    dp = device_packed(p, dev)
    w_want = oracle.decode_packed_bf16(p)
    gemv_option("gemv_strips", 1)
    gemv_option("gemv_tiles", 1 if kernel.startswith("tiles") else -1)
    gemv_option("gemv_tile_rows", {"tiles of 8": 3, "tiles of 4": 2}.get(kernel, 0))
    gemv_option("gemv_tile_cus", 2 if kernel.startswith("tiles of") else 0)
    cols = (0, 3, 4, 7, 8, 31, 32, 127, 128, 511, 512, 1023)
    if kernel == "tiles of 8":
        cols = cols[:8]
    if kernel == "tiles of 4":
        cols = cols[8:]
    x = torch.zeros(len(cols), in_f, dtype=torch.bfloat16)
    for i, k in enumerate(cols):
        x[i, k] = 1.0
    y = run_gemv(dp, 512, x, len(cols), dev)
    for i, k in enumerate(cols):
        assert np.array_equal(y[i], w_want[:, k]), (kind, k)


def test_gemv_is_reproducible(oracle, dev):
    p = make_packed("calibrated_odd_scale", 256, 2048)
    dp = device_packed(p, dev)
    x = activations(4, 2048, seed=5)
    first = run_gemv(dp, 512, x, 4, dev)
    for _ in range(5):
        assert np.array_equal(run_gemv(dp, 512, x, 4, dev), first)


@pytest.mark.parametrize("lanes", [True, False])
@pytest.mark.parametrize("shape", [(1536, 1536), (4608, 1536), (1536, 4608)])
def test_reference_call_surface(oracle, dev, shape, lanes):
    """fused_gemv / StreamingLinear called the way the reference's tests call them
    (tests/test_fused.py:24-33, tests/test_splitk.py:25-33), on the reference's weight recipe."""
    from ixrun_amd.engine import StreamingLinear
    from ixrun_amd.fused import compute_row_prefixes, fused_gemv, _pick_split

    out_f, in_f = shape
    p = quantize(outlier_weight(out_f, in_f, seed=0))
    x = activations(1, in_f, seed=1).reshape(in_f)
    y64 = oracle.gemm_f64(oracle.decode_packed_bf16(p), bf16_bits(x).reshape(1, -1))
    b1, b2 = (t.to(dev) for t in p["bitmaps"])
    l1, l2, l3 = (t.to(dev) for t in p["streams"])
    q1, q2 = compute_row_prefixes(p)
    y = fused_gemv(x.to(dev), b1, b2, l1, l2, l3, q1.to(dev), q2.to(dev), p["scale"].to(dev), out_f, in_f)
    assert y.dtype == torch.bfloat16 and y.shape == (out_f,)
    check_outputs(bf16_bits(y).reshape(1, -1), y64, f"fused_gemv {shape}")
    split = _pick_split(in_f) if out_f < in_f else 1
    if split > 1:
        chunk = in_f // split
        q1c, q2c = compute_row_prefixes(p, chunk)
        y32 = torch.zeros(out_f, dtype=torch.float32, device=dev)
        ret = fused_gemv(x.to(dev), b1, b2, l1, l2, l3, q1c.to(dev), q2c.to(dev), p["scale"].to(dev), out_f, in_f,
                         chunk=chunk, y32=y32)
        assert ret is y32
        check_outputs(y32.cpu().numpy().reshape(1, -1), y64, f"fused_gemv split {shape}")

    bias = torch.randn(out_f, generator=torch.Generator().manual_seed(3)).bfloat16()
    sl = StreamingLinear(p, bias=bias, lanes=lanes)
    shared = torch.empty(p["N"], dtype=torch.bfloat16, device=dev)
    sl._set_shared_buf(shared)
    assert np.array_equal(sl._q1.cpu().numpy(), (compute_row_prefixes(p, sl._split_chunk) if sl._split_chunk
                                                   else compute_row_prefixes(p))[0].numpy())
    w_ref = torch.from_numpy(oracle.decode_packed_bf16(p).view(np.int16)).view(torch.bfloat16)
    assert torch.equal(sl._decode().cpu(), w_ref)
    for xin in (x.to(dev).reshape(1, 1, in_f), activations(3, in_f, seed=2).to(dev), activations(40, in_f, seed=3).to(dev)):
        out = sl(xin)
        assert out.shape == xin.shape[:-1] + (out_f,) and out.dtype == torch.bfloat16
        want = torch.nn.functional.linear(xin.float().cpu(), w_ref.float()).double().numpy()
        got = (out.float().cpu() - bias.float()).double().numpy()
        assert rel_l2(got, want) < 6e-3  # bias add and output are bf16-rounded


@pytest.mark.parametrize("kind", ["outlier", "student_t", "rare_other", "only_l3"])
@pytest.mark.parametrize("level_bits", [(3, 5, 8), (3, 4, 5, 6, 8)])
def test_gemv_many_rows_to_a_workgroup(oracle, dev, kind, level_bits):
    """More rows than 256 workgroups hold at 64 apiece (16640 rows: 68 to a workgroup, in one round): the row-block
    kernel with row slots above 63, for one and two activation rows, dense mixes forced onto it as well (every lane
    with elements above level 1, the queue resolved inside the loop)."""
    from ixrun_amd import _lib

    out_f, in_f = 16640, 512
    p = make_packed(kind, out_f, in_f, level_bits)
    dp = device_packed(p, dev)
    w_bits = oracle.decode_packed_bf16(p)
    for m in (1, 2):
        x = activations(m, in_f, seed=m)
        y = run_gemv(dp, 512, x, m, dev, flags=_lib.IXH_GEMV_FORCE_358)
        check_outputs(y, oracle.gemm_f64(w_bits, bf16_bits(x)), f"{kind} {level_bits} {out_f}x{in_f} m={m}")


@pytest.fixture(scope="module", params=[True, False], ids=["lanes", "packed"])
def gate_up_layer(oracle, dev, request):
    """17408 x 5120 Student-t, packed once for its batch sizes, with the lane layout and without."""
    from ixrun_amd.engine import StreamingLinear

    p = quantize(student_t_weight(17408, 5120, seed=0))
    w_bits = oracle.decode_packed_bf16(p)
    return StreamingLinear(p, lanes=request.param), w_bits


@pytest.mark.parametrize("m", [1, 2, 4, 8, 16])
def test_full_size_config4_every_batch(oracle, dev, gate_up_layer, m):
    """17408 x 5120 with M in {2, 4, 8, 16} activation rows, and one row, each through the
    kernel the library picks for it (from the packed streams 1 and 2 rows: the row-block kernel, 68 rows to a workgroup;
    4, 8 and 16 rows: the tile kernel, at 16 rows with the activations in two column parts)."""
    sl, w_bits = gate_up_layer
    x = activations(m, 5120, seed=1)
    y = sl(x.to(dev))
    assert y.shape == (m, 17408)
    check_outputs(bf16_bits(y), oracle.gemm_f64(w_bits, bf16_bits(x)), f"17408x5120 m={m}")


@pytest.fixture(scope="module", params=[True, False], ids=["lanes", "packed"])
def down_proj_layer(oracle, dev, request):
    """The headline layer, 5120 x 17408 Student-t, packed once for several batch sizes, with lanes and without."""
    from ixrun_amd.engine import StreamingLinear

    p = quantize(student_t_weight(5120, 17408, seed=0))
    return StreamingLinear(p, lanes=request.param), oracle.decode_packed_bf16(p)


@pytest.mark.parametrize("m", [3, 6, 8, 9, 10, 12, 16, 24])
def test_full_size_down_proj_many_rows(oracle, dev, down_proj_layer, m):
    """5120 x 17408 with 3..16 activation rows as the library plans them on the whole device; from the packed streams
    20 rows to a workgroup at one or two activation rows; from three rows on blocks of 40 to 124 rows shared by two to six workgroups, each
    with a run of the column blocks (their sums added by a second launch); 24 rows in two calls."""
    sl, w_bits = down_proj_layer
    x = activations(m, 17408, seed=m)
    y = sl(x.to(dev))
    assert y.shape == (m, 5120)
    check_outputs(bf16_bits(y), oracle.gemm_f64(w_bits, bf16_bits(x)), f"5120x17408 m={m}")


def test_full_size_split_k_contract(oracle, dev):
    """The reference's split-K call on the headline shape (ixrun/engine.py:148-159: fused_gemv(..., chunk=8704, y32)
    on 5120 x 17408): the caller-zeroed fp32 vector comes back holding the sums, and a second call adds to it."""
    from ixrun_amd.fused import compute_row_prefixes, fused_gemv, _pick_split

    out_f, in_f = 5120, 17408
    p = quantize(student_t_weight(out_f, in_f, seed=0))
    assert _pick_split(in_f) == 2
    chunk = in_f // 2
    x = activations(1, in_f, seed=1).reshape(in_f)
    y64 = oracle.gemm_f64(oracle.decode_packed_bf16(p), bf16_bits(x).reshape(1, -1))
    b1, b2 = (t.to(dev) for t in p["bitmaps"])
    l1, l2, l3 = (t.to(dev) for t in p["streams"])
    q1c, q2c = compute_row_prefixes(p, chunk)
    y32 = torch.zeros(out_f, dtype=torch.float32, device=dev)
    args = (x.to(dev), b1, b2, l1, l2, l3, q1c.to(dev), q2c.to(dev), p["scale"].to(dev), out_f, in_f)
    ret = fused_gemv(*args, chunk=chunk, y32=y32)
    assert ret is y32
    once = y32.cpu().numpy().copy()
    check_outputs(once.reshape(1, -1), y64, "split-K 5120x17408")
    fused_gemv(*args, chunk=chunk, y32=y32)  # the contract is "add": a second call doubles every entry
    assert np.array_equal(y32.cpu().numpy(), once + once)


@pytest.mark.parametrize("lanes", [True, False])
def test_headline_kernel_is_reproducible(oracle, dev, lanes):
    """Repeat launches on a layer that is almost all level 1 (the headline workload, 5120 x 17408 Student-t; without lanes
    the row-block kernel) give the same bits, for one and for four activation rows."""
    from ixrun_amd.engine import StreamingLinear

    p = quantize(student_t_weight(5120, 17408, seed=0))
    assert p["counts"][0] >= 0.97 * p["N"]
    sl = StreamingLinear(p, lanes=lanes)
    for m in (1, 4):
        x = activations(m, 17408, seed=5).to(dev)
        first = bf16_bits(sl(x))
        for _ in range(5):
            assert np.array_equal(bf16_bits(sl(x)), first), m


@pytest.mark.parametrize("lanes", [True, False])
@pytest.mark.parametrize("shape,m", [((5120, 5120), 1), ((5120, 17408), 1), ((17408, 5120), 4)])
def test_full_size_layers(oracle, dev, shape, m, lanes):
    """The square, down and gate/up layers at full size: decoded int8 bit-exact, outputs within tolerance."""
    from ixrun_amd.engine import StreamingLinear

    out_f, in_f = shape
    w = student_t_weight(out_f, in_f, seed=0)
    p = quantize(w)
    q_want = oracle.decode_packed_i8(p)
    sl = StreamingLinear(p, lanes=lanes)
    o8 = torch.empty(p["N"], dtype=torch.int8, device=dev)
    sl._dp.decode(sl._table, sl._unit, out_i8=o8)
    assert np.array_equal(o8.cpu().numpy(), q_want)
    x = activations(m, in_f, seed=1)
    y = sl(x.to(dev))
    w_bits = oracle.dequant_bf16(q_want, oracle.packed_to_numpy(p)["scale_bits"]).reshape(out_f, in_f)
    # the bf16 decode as the library chooses it for this tensor (the row-block decoder: > 97 % level 1)
    o16 = torch.zeros(p["N"], dtype=torch.bfloat16, device=dev)
    sl._dp.decode(sl._table, sl._unit, out_bf16=o16)
    assert np.array_equal(bf16_bits(o16).reshape(out_f, in_f), w_bits)
    del o16
    y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
    err = check_outputs(bf16_bits(y), y64, f"full {shape} m={m}")
    print(f"{shape} m={m}: rel-L2 {err:.2e}, fractions {[round(c / p['N'], 5) for c in p['counts']]}, "
          f"packed {p['total_bytes']} B")


def test_full_size_five_level_decode(oracle, dev):
    """5120 x 17408 Student-t in the five-level scheme: the bf16 decode (row-block decoder, elements above level 1
    followed down four bitmaps) equals the oracle's, every element."""
    p = quantize(student_t_weight(5120, 17408, seed=0), (3, 4, 5, 6, 8))
    dp = device_packed(p, dev)
    table = dp.prefix_build(512)
    o16 = torch.zeros(p["N"], dtype=torch.bfloat16, device=dev)
    dp.decode(table, 512, out_bf16=o16)
    assert np.array_equal(bf16_bits(o16), oracle.decode_packed_bf16(p).reshape(-1))


@pytest.mark.parametrize("lanes", [True, False])
def test_full_size_calibrated_layer(oracle, dev, lanes):
    """5120 x 17408 with the 55/40/5 level mix of real LLM weights: the any-scheme kernels on runs of more than
    eight table units per wave (GEMV pieces of 8-9 units, decode runs of 11), against the oracle."""
    from ixrun_amd.engine import StreamingLinear

    out_f, in_f = 5120, 17408
    w, _ = calibrated_weight(out_f, in_f, seed=0, scale=0.0123046875)
    p = quantize(w)
    sl = StreamingLinear(p, lanes=lanes)
    shared = torch.empty(p["N"], dtype=torch.bfloat16, device=dev)
    sl._set_shared_buf(shared)
    w_bits = oracle.decode_packed_bf16(p)
    assert np.array_equal(bf16_bits(sl._decode()), w_bits)
    # (without lanes) two rows: weights gathered per wave; eight and sixteen: the matrix-pipe kernel (a row block's spans lie in two
    # workgroups here: 320 blocks of 16 rows x 9 spans dealt to one workgroup per CU)
    for m in (2, 8, 16):
        x = activations(m, in_f, seed=m)
        y = sl(x.to(dev))
        y64 = oracle.gemm_f64(w_bits, bf16_bits(x))
        check_outputs(bf16_bits(y), y64, f"full-size calibrated m={m}")


@pytest.mark.parametrize("n_units", [1, 127, 128, 129, 384, 1025])
@pytest.mark.parametrize("level_bits,chunk", [((3, 5, 8), 512), ((2, 8), 5), ((3, 4, 5, 6, 8), 777), ((1, 2, 3, 4, 5, 6, 7, 8), 33)])
def test_prefix_build_with_and_without_a_workspace(oracle, dev, n_units, level_bits, chunk):
    """Both builders against the oracle, around the 128 units of a tile, with the last unit cut short."""
    import ctypes as C

    from ixrun_amd import _lib

    n = n_units * chunk - chunk // 2
    p = make_packed("student_t", 1, n, level_bits)
    dp = device_packed(p, dev)
    want = oracle.prefix(n, len(level_bits), [b.numpy().view(np.uint32) for b in p["bitmaps"]], chunk)
    assert np.array_equal(dp.prefix_build(chunk).cpu().numpy(), want)
    plain = torch.full_like(torch.from_numpy(want), -1).to(dev)
    _lib.check(_lib.lib().ixh_prefix_build(C.byref(dp.struct), chunk, plain.data_ptr(), _lib.current_stream(dev)))
    assert np.array_equal(plain.cpu().numpy(), want)
    rc = _lib.lib().ixh_prefix_build_ws(C.byref(dp.struct), chunk, plain.data_ptr(), plain.data_ptr(), 0, None)
    assert rc == -4, "a workspace that is too small"
