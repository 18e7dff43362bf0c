"""Device decode of the group-scale format (ixh_decode_gs) against the CPU oracle: bf16 bit patterns must be equal.
Mirrors the reference's ixgs/test_gs.py on the GPU path."""
import numpy as np
import pytest
import torch

from helpers import bf16_bits, int8_mix, packed_from_int8
from test_ixgs_cpu import heavy_tail

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from ixrun_amd import _lib

    assert _lib.lib().ixh_version() >= 100
    return torch.device("cuda:0")


def packed_from_ints(oracle, q, scales, out_f, in_f, group):
    """A packed dictionary straight from integers, for values the quantizer never produces (tier 3, +128)."""
    e = oracle.gs_encode(q)
    i32 = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int32).copy())
    n2, n3 = e["counts"][1], e["counts"][2]
    return {"out_f": out_f, "in_f": in_f, "N": out_f * in_f, "group_size": group,
            "group_scales": torch.from_numpy(scales.view(np.float16).copy()),
            "b1": i32(e["b1"]), "b2": i32(e["b2"]) if n2 + n3 else torch.zeros(1, dtype=torch.int32),
            "l1": i32(e["l1"]), "l2": i32(e["l2"]),
            "l3": torch.from_numpy(e["l3"].copy()) if n3 else torch.zeros(1, dtype=torch.uint8),
            "counts": e["counts"], "total_bytes": 0, "bits_per_weight": 0.0, "compression_vs_bf16": 0.0}


@pytest.fixture(params=["by_mix", "staged", "dense"])
def decoder(request, force_decoder):
    """Which of the two unit-512 decoders runs: chosen by the mix of tiers, or forced (level by level where the
    group size allows it, or the one that stages the streams)."""
    if request.param != "by_mix":
        force_decoder(request.param)
    return request.param


@pytest.mark.parametrize("shape,group", [((512, 256), 64), ((1000, 640), 64), ((1, 1), 64), ((3, 11), 64), ((33, 1000), 64),
                                         ((300, 1031), 64), ((256, 4608), 64), ((128, 512), 8), ((128, 512), 32),
                                         ((64, 1536), 128), ((40, 100), 20), ((7, 513), 3), ((2048, 2048), 64)])
def test_decode_matches_oracle(oracle, dev, decoder, shape, group):
    from ixrun_amd import ixgs

    w = heavy_tail(shape, seed=1)
    p = ixgs.int8gs_quantize(w, group)
    scales, q = oracle.gs_quantize(bf16_bits(w), group)
    want = oracle.gs_dequant_bf16(q, scales, group)
    got = ixgs.decode_weight_triton(p, dev)
    assert got.shape == tuple(shape) and got.dtype == torch.bfloat16
    assert np.array_equal(bf16_bits(got).reshape(-1), want)
    assert torch.equal(got.cpu(), ixgs.decode_weight_scatter(p, device="cpu"))  # ixgs/test_gs.py:61-75


@pytest.mark.parametrize("mix", ["all_tiers", "only_tier3", "only_tier2", "dense_mix"])
@pytest.mark.parametrize("shape,group", [((64, 1536), 64), ((37, 1000), 64), ((5, 100), 10)])
def test_decode_hand_built_tiers(oracle, dev, decoder, mix, shape, group):
    """Integers over the whole range [-127, 128], which the quantizer itself never emits."""
    from ixrun_amd import ixgs

    n = shape[0] * shape[1]
    rng = np.random.default_rng(7)
    if mix == "all_tiers":
        q = rng.integers(-3, 5, size=n)
        r = rng.random(n)
        q[r < 0.3] = rng.integers(-15, 17, size=int((r < 0.3).sum()))
        q[r < 0.05] = rng.integers(-127, 129, size=int((r < 0.05).sum()))
        q[:4] = [128, -127, 16, -15]
    elif mix == "only_tier3":
        q = rng.choice([-127, -100, -16, 17, 99, 128], size=n)
    elif mix == "only_tier2":
        q = rng.choice([-15, -4, 5, 16], size=n)
    else:
        q = rng.integers(-127, 129, size=n)
    q = q.astype(np.int16)
    scales = (rng.random(-(-n // group)).astype(np.float32) * 0.01 + 1e-4).astype(np.float16).view(np.uint16)
    p = packed_from_ints(oracle, q, scales, shape[0], shape[1], group)
    got = ixgs.decode_weight_triton(p, dev)
    assert np.array_equal(bf16_bits(got).reshape(-1), oracle.gs_dequant_bf16(q, scales, group))


def on_device(p, dev):
    return {k: v.to(dev) if isinstance(v, torch.Tensor) else v for k, v in p.items()}


@pytest.mark.parametrize("mix", ["only_tier1", "only_tier2", "only_tier3", "all_tiers", "tier2_first"])
@pytest.mark.parametrize("n", [1, 31, 32, 2047, 2048, 2049, 2048 * 256, 2048 * 256 + 1, 2048 * 1500 + 77, (1 << 22) - 5, 1 << 22])
def test_decode_without_a_table(oracle, dev, mix, n):
    """One launch, whose workgroups count the bitmaps in front of them: the edges of a word, a span, a span a workgroup, and the
    largest size; bitmap 1 empty, full and of its own density."""
    from ixrun_amd import _lib, ixgs
    import ctypes as C

    rng = np.random.default_rng(n)
    q = {"only_tier1": rng.integers(-3, 5, size=n), "only_tier2": rng.choice([-15, -4, 5, 16], size=n),
         "only_tier3": rng.choice([-127, -16, 17, 128], size=n), "all_tiers": rng.integers(-3, 5, size=n),
         "tier2_first": rng.integers(-3, 5, size=n)}[mix].astype(np.int16)
    if mix == "all_tiers":
        r = rng.random(n)
        q[r < 0.45] = rng.integers(-15, 17, size=int((r < 0.45).sum()))
        q[r < 0.05] = rng.integers(-127, 129, size=int((r < 0.05).sum()))
    if mix == "tier2_first":
        q[: n // 3] = 16
        q[n // 3 : n // 3 + 5] = 128
    scales = (rng.random(-(-n // 64)).astype(np.float32) * 0.01 + 1e-4).astype(np.float16).view(np.uint16)
    p = on_device(packed_from_ints(oracle, q, scales, 1, n, 64), dev)
    want = oracle.gs_dequant_bf16(q, scales, 64)
    dp = _lib.DevicePacked((3, 5, 8), 1, n, [p["b1"], p["b2"]], [p["l1"], p["l2"], p["l3"]], None)
    out = torch.full((n + 8,), 7.0, dtype=torch.bfloat16, device=dev)
    _lib.check(_lib.lib().ixh_decode_unranked(C.byref(dp.struct), p["group_scales"].data_ptr(), 64, out.data_ptr(), _lib.current_stream(dev)))
    assert np.array_equal(bf16_bits(out)[:n], want) and bool((out[n:] == 7.0).all())
    assert np.array_equal(bf16_bits(ixgs.decode_weight_triton(p)).reshape(-1), want)


@pytest.mark.parametrize("kind", ["only_l1", "no_l3", "no_l2", "only_l3", "rare_other"])
@pytest.mark.parametrize("shape", [(1, 1), (3, 683), (33, 1000), (700, 1031)])
def test_per_tensor_decode_without_a_table(oracle, dev, kind, shape):
    from ixrun_amd import _lib, decode_weight_triton
    import ctypes as C

    out_f, in_f = shape
    p = packed_from_int8(int8_mix(kind, out_f * in_f, seed=3), out_f, in_f)
    want = oracle.decode_packed_bf16(p).reshape(-1)
    dp = _lib.DevicePacked.from_dict(p, dev)
    out = torch.empty(out_f * in_f, dtype=torch.bfloat16, device=dev)
    _lib.check(_lib.lib().ixh_decode_unranked(C.byref(dp.struct), None, 0, out.data_ptr(), _lib.current_stream(dev)))
    assert np.array_equal(bf16_bits(out), want)
    assert np.array_equal(bf16_bits(decode_weight_triton(p)).reshape(-1), want)


@pytest.mark.parametrize("mix", ["tier1", "tier3", "all"])
@pytest.mark.parametrize("n", [(1 << 21) + 1, 256 * 5 * 2048 - 31, 256 * 5 * 2048, 256 * 7 * 2048 + 4096 + 33, (1 << 22) - 127, 1 << 22])
def test_bitmaps_counted_by_a_launch_of_their_own(oracle, dev, n, mix):
    """Workgroups that begin within a run of counted words and at one; either bitmap whole and next to empty; one launch gives the same."""
    from ixrun_amd import _lib
    import ctypes as C

    rng = np.random.default_rng(n)
    q = {"tier1": rng.integers(-3, 5, size=n), "tier3": rng.choice([-127, -16, 17, 128], size=n), "all": rng.integers(-20, 21, size=n)}[mix].astype(np.int16)
    q[n // 2] = 9
    scales = (rng.random(-(-n // 64)).astype(np.float32) * 0.01 + 1e-4).astype(np.float16).view(np.uint16)
    p = on_device(packed_from_ints(oracle, q, scales, 1, n, 64), dev)
    dp = _lib.DevicePacked((3, 5, 8), 1, n, [p["b1"], p["b2"]], [p["l1"], p["l2"], p["l3"]], None)
    need = _lib.lib().ixh_decode_unranked_workspace_bytes(C.byref(dp.struct))
    assert need > 0
    out, one = (torch.full((n + 8,), 7.0, dtype=torch.bfloat16, device=dev) for _ in range(2))
    ws = torch.full((need + 64,), 0xA5, dtype=torch.uint8, device=dev)
    call = lambda ws_ptr, given: _lib.lib().ixh_decode_unranked_ws(C.byref(dp.struct), p["group_scales"].data_ptr(), 64, out.data_ptr(), ws_ptr, given,
                                                                   _lib.current_stream(dev))
    assert call(None, need) == call(ws.data_ptr(), need - 1) == call(ws.data_ptr() + 2, need) == -4
    for _ in range(2):
        _lib.check(call(ws.data_ptr(), need))
    _lib.check(_lib.lib().ixh_decode_unranked(C.byref(dp.struct), p["group_scales"].data_ptr(), 64, one.data_ptr(), _lib.current_stream(dev)))
    assert np.array_equal(bf16_bits(out)[:n], oracle.gs_dequant_bf16(q, scales, 64)) and bool((out[n:] == 7.0).all())
    assert torch.equal(out, one) and bool((ws[need:] == 0xA5).all())


def test_small_tensors_are_counted_in_one_launch(dev):
    from ixrun_amd import _lib
    import ctypes as C

    for out_f, in_f, counted in ((1 << 10, 1 << 11, 0), (1 << 11, 1 << 11, 1), ((1 << 11) + 1, 1 << 11, 0)):
        s = _lib.IxhPacked(n_levels=3, out_f=out_f, in_f=in_f)
        assert (_lib.lib().ixh_decode_unranked_workspace_bytes(C.byref(s)) > 0) == bool(counted)


@pytest.mark.parametrize("levels,shape", [((3, 4, 5, 6, 8), (33, 1000)), ((3, 5, 8), (2049, 2048))])
def test_a_decode_that_succeeds_leaves_no_error(oracle, dev, levels, shape):
    """Tensors that need a table are not first refused without one."""
    from ixrun_amd import _lib, decode_weight_triton
    from ixrun_amd.quantize import int8x_quantize_device

    w = (torch.randn(shape, generator=torch.Generator().manual_seed(5)) * 0.02).bfloat16().to(dev)
    p = int8x_quantize_device(w, levels)
    p.pop("table512", None)
    assert _lib.lib().ixh_set_option(b"no such option", 0) == -1
    before = _lib.lib().ixh_last_error()
    got = decode_weight_triton(p)
    assert _lib.lib().ixh_last_error() == before
    on_host = lambda v: v.cpu() if isinstance(v, torch.Tensor) else [on_host(e) for e in v] if isinstance(v, list) else v
    host = {k: on_host(v) for k, v in p.items()}
    assert np.array_equal(bf16_bits(got), oracle.decode_packed_bf16(host).reshape(shape))


@pytest.mark.parametrize("n,group,code", [((1 << 22) + 1, 64, -2), (4096, 48, -2), (4096, 16, -2), (4096, 0, -1)])
def test_decode_without_a_table_refuses_the_rest(oracle, dev, n, group, code):
    from ixrun_amd import _lib
    import ctypes as C

    p = on_device(packed_from_ints(oracle, np.zeros(n, dtype=np.int16), np.ones(n, dtype=np.uint16), 1, n, group), dev)
    dp = _lib.DevicePacked((3, 5, 8), 1, n, [p["b1"], p["b2"]], [p["l1"], p["l2"], p["l3"]], None)
    out = torch.full((n,), 7.0, dtype=torch.bfloat16, device=dev)
    assert _lib.lib().ixh_decode_unranked(C.byref(dp.struct), p["group_scales"].data_ptr(), group, out.data_ptr(), _lib.current_stream(dev)) == code
    assert bool((out == 7.0).all())


def test_linear_and_deploy(oracle, dev):
    from ixrun_amd import ixgs

    w = heavy_tail((256, 128), seed=2)
    x = torch.randn(8, 128, generator=torch.Generator("cpu").manual_seed(2)).bfloat16().to(dev)
    p = ixgs.int8gs_quantize(w)
    for cache in ("full", "none"):
        layer = ixgs.Int8GSLinear(p, cache=cache)
        want = torch.nn.functional.linear(x, ixgs.decode_weight_scatter(p, dev))
        assert torch.equal(layer(x), want)
    model = torch.nn.Sequential(torch.nn.Linear(128, 256), torch.nn.GELU(), torch.nn.Linear(256, 64)).bfloat16()
    with torch.no_grad():
        model[0].weight.copy_(w)
    ref = model.to(dev)(x)
    import copy

    deployed = copy.deepcopy(model)
    stats = ixgs.deploy_model_gs(deployed, verbose=False)
    assert stats["n_layers"] == 2 and isinstance(deployed[0], ixgs.Int8GSLinear) and stats["counts"][2] == 0
    out = deployed.to(dev)(x)
    corr = torch.corrcoef(torch.stack([ref.float().flatten(), out.float().flatten()]))[0, 1]
    assert corr > 0.99


def test_rejects_bad_arguments(dev):
    from ixrun_amd import _lib, ixgs

    p = ixgs.int8gs_quantize(heavy_tail((8, 64), seed=0))
    mv = lambda t: t.to(dev)
    dp = _lib.DevicePacked((3, 5, 8), 8, 64, [mv(p["b1"]), mv(p["b2"])], [mv(p["l1"]), mv(p["l2"]), mv(p["l3"])], None)
    table = dp.prefix_build(512)
    out = torch.empty(512, dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError):
        dp.decode_gs(table, 512, mv(p["group_scales"])[:3], 64, out)
    with pytest.raises(_lib.IxhError):
        dp.decode_gs(table, 512, mv(p["group_scales"]), 0, out)
