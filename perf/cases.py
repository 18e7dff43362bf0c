"""What the framework is timed on: packed linear layers as a program that serves a model calls them, and the decode and
encode calls around them.

A case names one operation, its layer shape, the level scheme and the mix of weights:

  op "linear"     StreamingLinear.forward of one deployed layer; `rows` activation rows (1: a token; 2 .. 16: a batch of
                  token streams; more: a prompt)
  op "block"      the linear layers of one transformer block, one token, replayed from a captured graph
  op "decode"     decode_weight_triton: the whole bf16 weight from a packed dictionary (Int8XLinear with cache="none"
                  calls it in each forward)
  op "encode"     int8x_quantize_device: quantise and pack a bf16 weight (each layer of a deploy)
  op "gs_decode"  ixgs.decode_weight_triton: the group-scale sibling format

  mix "real"      integers in the levels of (3,5,8) at 55 / 40 / 5 %, the fractions of trained weights
  mix "t"         Student-t weights (nu = 4), the benchmark's recipe: nearly all in the first level on a large layer
  mix "outlier"   N(0, 0.005) with 4 % N(0, 0.05)
"""
from __future__ import annotations

import math

import torch

from ixrun_amd import Int8XEngine, decode_weight_triton, ixgs
from ixrun_amd.quantize import int8x_quantize_device

DEV = "cuda"
SCHEMES = {"358": (3, 5, 8), "34568": (3, 4, 5, 6, 8)}
# (out_f, in_f) of the block's layers: mixer input, mixer output, gate, up, down
BLOCK = ((10240, 5120), (5120, 5120), (17408, 5120), (17408, 5120), (5120, 17408))
MOST_WEIGHTS = 5120 * 17408
MOST_PRODUCTS = MOST_WEIGHTS * 512


def _linear(name, out_f, in_f, rows, mix, scheme="358", bias=False):
    return {"name": name, "op": "linear", "out_f": out_f, "in_f": in_f, "rows": rows, "mix": mix, "scheme": scheme,
            "bias": bias}


def listed():
    return [
        # the smallest call: one token through a small projection with a bias, where launches and the host path count
        _linear("token_small", 1536, 1536, 1, "outlier", bias=True),
        # the benchmark's headline: one token through a large layer that is nearly all first level
        _linear("token_t", 5120, 17408, 1, "t"),
        # a token through all linear layers of a block, weights mixed as trained ones are, from a captured graph
        {"name": "token_block_graph", "op": "block", "mix": "real", "scheme": "358"},
        # the denser five-level scheme on the same weights
        _linear("token_five", 17408, 5120, 1, "real", "34568"),
        # rows that are no whole number of 512-element units
        _linear("token_odd", 4096, 11008, 1, "real"),
        # several token streams served together
        _linear("batch8", 17408, 5120, 8, "real"),
        _linear("batch16_t", 5120, 17408, 16, "t"),
        # prompts: a short one of an odd length, and the benchmark's 512 rows in five levels
        _linear("prompt_short", 10240, 5120, 100, "real"),
        _linear("prompt_512", 5120, 17408, 512, "t", "34568"),
        # the whole weight, as a cache="none" forward or a load-time decode asks for it
        {"name": "decode", "op": "decode", "out_f": 17408, "in_f": 5120, "mix": "real", "scheme": "358"},
        # packing one layer of a deploy
        {"name": "encode", "op": "encode", "out_f": 5120, "in_f": 17408, "mix": "real", "scheme": "358"},
        # the group-scale format; its writer runs on the host, which bounds the size here
        {"name": "gs_decode", "op": "gs_decode", "out_f": 2048, "in_f": 2048, "mix": "t", "scheme": "358", "group": 64},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, kind):
    v = _log(rng, lo, hi)
    step = {"unit": 512, "word": 32, "any": 1}[kind]
    return max(step, min(int(round(v / step)) * step, hi // step * step))


def draw(rng):
    """Shapes from 256 to 17408 a side. Rows of whole 512-element units as most models have them, of whole 32-bit words,
    and now and then of any length."""
    op = rng.choice(("linear",) * 6 + ("decode", "encode", "gs_decode"))
    big = 2048 if op == "gs_decode" else 17408
    in_f = _size(rng, 512, big, rng.choice(("unit",) * 5 + ("word",) * 3 + ("any",)))
    out_f = _size(rng, 256, min(big, max(256, MOST_WEIGHTS // in_f)), rng.choice(("word", "word", "any")))
    mix = rng.choice(("real", "real", "t", "outlier"))
    case = {"op": op, "out_f": out_f, "in_f": in_f, "mix": mix, "scheme": "358"}
    if op == "gs_decode":
        case["group"] = rng.choice((32, 64, 64, 128))
        return case
    case["scheme"] = rng.choice(("358", "358", "358", "34568"))
    if op == "linear":
        rows = rng.choice((1, 1, 0, 0, 17))
        if rows == 0:
            rows = int(round(_log(rng, 2, 16)))
        elif rows == 17:
            rows = int(round(_log(rng, 17, max(17, min(1024, MOST_PRODUCTS // (out_f * in_f))))))
        case["rows"] = rows
        case["bias"] = rng.random() < 0.25
    return case


# ---------------------------------------------------------------------------------------------------------------------
#  weights
# ---------------------------------------------------------------------------------------------------------------------
def _weight(out_f, in_f, mix, gen):
    n = out_f * in_f
    if mix == "t":  # scaled to a standard deviation of 0.02
        z = torch.randn(n, generator=gen, device=DEV)
        chi = torch.randn(n, generator=gen, device=DEV).square_()
        for _ in range(3):
            chi += torch.randn(n, generator=gen, device=DEV).square_()
        w = z.div_(chi.div_(4).sqrt_())
        # the largest weight sets the scale and so the level shares: its median, so that these hang on the size alone
        top = _t_largest(n)
        w.clamp_(-top, top)
        w[int(torch.randint(n, (1,), generator=gen, device=DEV))] = top
        w.mul_(0.02 / 2 ** 0.5)
    elif mix == "outlier":
        w = torch.randn(n, generator=gen, device=DEV).mul_(0.005)
        far = torch.rand(n, generator=gen, device=DEV) < 0.04
        w = torch.where(far, torch.randn(n, generator=gen, device=DEV).mul_(0.05), w)
    else:  # levels drawn, magnitudes uniform within a level; one 127 fixes the scale at a bf16 value that rounds
        u = torch.rand(n, generator=gen, device=DEV)
        f = torch.rand(n, generator=gen, device=DEV)
        w = torch.where(u < 0.55, (f * 4).floor_(), torch.where(u < 0.95, (f * 12).floor_() + 4, (f * 112).floor_() + 16))
        w.mul_((torch.rand(n, generator=gen, device=DEV) < 0.5).mul(2).sub(1))
        w[int(torch.randint(n, (1,), generator=gen, device=DEV))] = 127
        w.mul_(0.0019073486328125)  # 125 * 2**-16
    return w.to(torch.bfloat16).view(out_f, in_f)


def _t_tail(t):
    """P(|T| > t) for four degrees of freedom."""
    q = t * t / (1 + t * t / 4)
    return 1 - 0.75 * math.sqrt(q) * (1 - q / 12)


def _t_largest(n):
    """The median of the largest |T| of n."""
    lo, hi = 1.0, 1e4
    for _ in range(60):
        mid = math.sqrt(lo * hi)
        lo, hi = (mid, hi) if n * _t_tail(mid) > math.log(2) else (lo, mid)
    return lo


def _beyond(case, edge):
    """Expected share of weights whose |integer| is above `edge`."""
    n, a = case["out_f"] * case["in_f"], edge + 0.5
    if case["op"] == "gs_decode":
        return 0.0 if edge >= 15 else 1 - a / 15 * 0.9
    if case["mix"] == "real":
        return 0.05 * (127 - edge) / 112 if edge >= 15 else 0.05 + 0.4 * (15 - edge) / 12
    if case["mix"] == "outlier":
        far = max(0.04 * n, 2.0)
        s = 0.05 * math.sqrt(2 * math.log(far)) / 127
        return 0.96 * math.erfc(a * s / 0.005 / math.sqrt(2)) + 0.04 * math.erfc(a * s / 0.05 / math.sqrt(2))
    return _t_tail(a * _t_largest(n) / 127)


def _packed_bytes(case):
    bits, left = 0.0, 1.0
    for b in SCHEMES[case["scheme"]][:-1]:
        rest = _beyond(case, (1 << (b - 1)) - 1)
        bits += left + (left - rest) * b
        left = rest
    n = case["out_f"] * case["in_f"]
    return n * (bits + 8 * left) / 8 + (2 * n / case["group"] if "group" in case else 2)


# ---------------------------------------------------------------------------------------------------------------------
#  the program around the calls
# ---------------------------------------------------------------------------------------------------------------------
def _deployed(shapes, case, gen):
    """The layers as a streaming deploy leaves them, with their shared decode buffer."""
    bias = bool(case.get("bias", False))
    layers = []
    for out_f, in_f in shapes:
        lin = torch.nn.Linear(in_f, out_f, bias=bias, device="meta", dtype=torch.bfloat16)
        lin.weight = torch.nn.Parameter(_weight(out_f, in_f, case["mix"], gen), requires_grad=False)
        if bias:
            b = torch.randn(out_f, generator=gen, device=DEV).mul_(0.02).to(torch.bfloat16)
            lin.bias = torch.nn.Parameter(b, requires_grad=False)
        layers.append(lin)
    model = torch.nn.ModuleList(layers)
    Int8XEngine._deploy_streaming(model, SCHEMES[case["scheme"]], verbose=False)
    return model


def _activations(rows, in_f, gen):
    shape = (rows, 1, in_f) if rows <= 16 else (1, rows, in_f)
    return torch.randn(shape, generator=gen, device=DEV).to(torch.bfloat16)


@torch.no_grad()
def prepare(case, seed):
    gen = torch.Generator(DEV).manual_seed(seed)
    op = case["op"]
    state = {"op": op}
    if op == "linear":
        state["layer"] = _deployed([(case["out_f"], case["in_f"])], case, gen)[0]
        state["x"] = _activations(case["rows"], case["in_f"], gen)
    elif op == "block":
        layers = _deployed(BLOCK, case, gen)
        xs = [_activations(1, in_f, gen) for _, in_f in BLOCK]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for layer, x in zip(layers, xs):
                layer(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ys = [layer(x) for layer, x in zip(layers, xs)]
        state.update(layers=layers, xs=xs, ys=ys, graph=graph)
    else:
        if op == "encode":
            # the stream lengths follow from the values: the same ones in an order of the seed's, so that they stay
            w = _weight(case["out_f"], case["in_f"], case["mix"], torch.Generator(DEV).manual_seed(0))
            w = w.view(-1)[torch.randperm(w.numel(), generator=gen, device=DEV)].view(w.shape)
            state.update(weight=w, levels=SCHEMES[case["scheme"]])
            return state
        w = _weight(case["out_f"], case["in_f"], case["mix"], gen)
        if op == "decode":
            state["packed"] = int8x_quantize_device(w, SCHEMES[case["scheme"]])
        else:
            packed = ixgs.int8gs_quantize(w, case["group"])
            state["packed"] = {k: v.to(DEV) if isinstance(v, torch.Tensor) else v for k, v in packed.items()}
    return state


@torch.no_grad()
def run(state):
    op = state["op"]
    if op == "linear":
        return state["layer"](state["x"])
    if op == "block":
        state["graph"].replay()
        return state["ys"]
    if op == "decode":
        return decode_weight_triton(state["packed"])
    if op == "gs_decode":
        return ixgs.decode_weight_triton(state["packed"])
    p = int8x_quantize_device(state["weight"], state["levels"])
    return {k: p[k] for k in ("scale", "bitmaps", "streams", "counts", "table512")}


def work(case):
    op = case["op"]
    shapes = BLOCK if op == "block" else ((case["out_f"], case["in_f"]),)
    nbytes = flops = 0.0
    for out_f, in_f in shapes:
        n = out_f * in_f
        one = dict(case, out_f=out_f, in_f=in_f)
        nbytes += _packed_bytes(one)
        if op in ("linear", "block"):
            rows = case.get("rows", 1)
            nbytes += 2 * rows * (in_f + out_f) + (2 * out_f if case.get("bias") else 0)
            flops += 2.0 * rows * n
        else:
            nbytes += 2 * n  # the bf16 weight, written or read
        if op == "encode":
            nbytes += 4 * (len(SCHEMES[case["scheme"]]) - 1) * (-(-n // 512) + 1)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bf16 outputs of fp32 sums taken in another order: a value may land on the neighbouring bf16, twice with a bias
    if case["op"] in ("linear", "block"):
        return {"rel": 4e-3, "max": 2e-2}
    return "exact"
