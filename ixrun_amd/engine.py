"""Deploy modules and engine of the INT8-X streaming path.

``StreamingLinear`` keeps a layer's packed streams resident on the GPU and
serves every forward from them: up to 16 activation rows go through the fused
decode+GEMV kernel (the bf16 weight never reaches memory), prompts of up to 256
to 1024 rows through a fused decode+GEMM, larger ones are decoded into a shared
bf16 buffer and multiplied with ``F.linear``.
``GraphLinear`` / ``Int8XEngine`` follow the reference's ``ixrun/engine.py``
(``StreamingLinear`` ``:40-173``, ``GraphLinear`` ``:179-196``,
``ResourceScheduler`` ``:202-235``, ``Int8XEngine`` ``:241-516``) and keep its
attribute names (``_b1 .. _l3, _scale, _b1_blk, _b2_blk, _q1, _q2,
_split_chunk, _use_fused, _w_buf``), which callers of ``fused_gemv`` read.
"""
from __future__ import annotations

import gc
import os

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad

from . import _lib, gemm_tuning
from .config import TRITON_BLOCK
from .fused import FUSED_TILE, _pick_split, _workspaces, pick_unit, shared_workspace
from .linear import _set_parent_child, iter_quantizable_linears
from .quantize import int8x_quantize, portable_packed, quantize_for_deploy

__all__ = ["Int8XEngine", "StreamingLinear", "GraphLinear", "ResourceScheduler"]

try:  # the current stream's handle and the current device, without building a Stream object (1 us less per forward)
    _raw_stream = torch._C._cuda_getCurrentRawStream
except AttributeError:  # pragma: no cover
    def _raw_stream(index):
        return torch.cuda.current_stream(index).cuda_stream
try:
    _current_device = torch._C._cuda_getDevice
except AttributeError:  # pragma: no cover
    _current_device = torch.cuda.current_device

LANE_BUFFERS = ("_lane_plane", "_lane_off", "_lane_pos", "_lane_val")
MAX_FUSED_ROWS = 16  # activation rows served by the fused decode+GEMV kernel
# With a decode buffer at hand, more rows than this go through decode + library GEMM.  Tensors that are almost all
# level 1, MI355X: the pair takes 72-75 us on 17408 x 5120 and 5120 x 17408 at any M up to 32 and 34-50 us on
# 5120 x 5120 (five levels: 73-74 and 38-39 us); the fused kernels take 25 / 27 us (17408 x 5120), 27 / 30 us
# (5120 x 17408) and 15 / 18 us (5120 x 5120) at M = 8 / 16 (five levels, measured before several workgroups could share
# a block of rows: 29 / 32, 39 / 51 and 23 / 31 us): every row count the fused kernels take.  Dense mixes (55 / 40 / 5 %): the pair takes
# 91-93 us on the large layers and 34-52 us on 5120 x 5120, the fused kernels 54-62 / 69-73 / 79-85 / 80-85 / 83-88 us
# (large layers) and 21 / 26 / 29 / 29 / 31 us (5120 x 5120) at M = 1 / 2 / 4 / 8 / 16: every row count as well.  Dense
# five-level mixes: one row 97-105 us fused against 120 us for the pair; two to sixteen rows 113-126 us fused (the
# decoder in its tile mode) against 119-123 us: the pair keeps those (the any-scheme kernel took 209-260 us).
MAX_FUSED_ROWS_WITH_BUFFER = 16
MAX_FUSED_ROWS_WITH_BUFFER_DENSE = 16
# 17 .. 32 rows on a large layer that is almost all level 1: two fused calls (16 rows and the rest) instead of the
# many-row paths.  MI355X, Student-t weights with 99.4 % of the elements in level 1, hipGraph replays over distinct
# layers: 5120 x 17408 at 17 / 24 / 32 rows 60 / 70 / 75 us in two calls against 118-120 us fused decode+GEMM and
# 137 us decode + library GEMM; 17408 x 5120 54 / 60 / 64 us against 120-122 and 87 us.  On 5120 x 5120 the two
# calls tie with the fused decode+GEMM (37-45 against 44-45 us) and lose to decode + library GEMM (34 us), and three
# calls for 33 .. 48 rows gain nothing on any shape: large layers and up to 32 rows only.  (A layer with lanes takes
# them in one pass instead, 5120 x 17408 27-28 us, unless its rows are no whole 16-byte pieces: _lanes_gemm_wins.)
SPLIT_FUSED_MIN_WEIGHTS = 40_000_000
# More rows than that: with a shared decode buffer the layer decodes into it and calls the library GEMM
# (5120 x 5120 five-level on MI355X: 60 us at 32 rows, 84 us at 512); without one it runs the fused
# decode+GEMM, which keeps the bf16 weight out of HBM altogether but is slower (84 us and 194 us): its
# decode shares the CU with the matrix-core tiles at two waves per SIMD, the stand-alone decode runs at six.


def _plain_call(x) -> bool:
    """Whether a product of ``x`` that is not torch's own is what the caller gets from ``F.linear``: no gradient, transform,
    other result type or other kind of tensor is asked for."""
    return (not (x.requires_grad and torch.is_grad_enabled()) and forward_ad._current_level < 0
            and not torch.overrides.has_torch_function_unary(x)
            and torch._C._functorch.peek_interpreter_stack() is None
            and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") is torch.bfloat16))


def _lane_bytes(level_bits, out_f, in_f, counts) -> int:
    """Bytes of a layer's lane layout, to within the unevenness of its rows; 0 where it would take more than the bf16 weight
    (see ``StreamingLinear._make_lanes``)."""
    n_bytes = _lib.LanePacked.estimate(level_bits, out_f, in_f, counts) or 0
    return n_bytes if n_bytes <= 2 * out_f * in_f else 0


class StreamingLinear(nn.Module):
    """GPU-resident packed weight, decoded inside every forward.

    Construction mirrors the reference (``ixrun/engine.py:49-104``): the packed
    tensors become buffers on the GPU and the rank tables are derived once.
    Here the tables are counted on the device from the bitmaps
    (``ixh_prefix_build``); ``_q1``/``_q2`` and ``_b1_blk``/``_b2_blk`` are the
    reference-shaped views of them.  Any level scheme is accepted; bitmaps and
    streams beyond the third level are registered as ``_b3``, ``_l4`` and so on.

    With ``lanes`` the same integers are kept in the lane layout as well
    (``csrc/ixh_lanes.h``; 3.1 to 6.5 bits a weight for the mixes that take 4.0
    to 5.5 packed), which the forwards of up to 16 rows and of most prompts
    read: one row of 5120 x 17408 takes 13.0 us from it instead of 16.8 (99 %
    of the weights in level 1), 17.1 instead of 48.7 (55 / 40 / 5 %), five
    levels 17.1 instead of 86.  It is no part of the state dict.
    """

    def __init__(self, packed: dict, bias=None, lanes: bool = True):
        super().__init__()
        self.out_features = packed["out_f"]
        self.in_features = packed["in_f"]
        self.N = packed["N"]
        self.level_bits = tuple(packed["level_bits"])
        self.counts = packed["counts"]

        n_levels = len(self.level_bits)
        for i in range(n_levels - 1):
            self.register_buffer(f"_b{i + 1}", packed["bitmaps"][i].cuda())
        for i in range(n_levels):
            self.register_buffer(f"_l{i + 1}", packed["streams"][i].cuda())
        self.register_buffer("_scale", packed["scale"].reshape(()).cuda())
        self.register_buffer("_bias", bias.detach().clone().cuda() if bias is not None else None)
        self._gemv_flags = 0  # extra IXH_GEMV_* flags of every fused call (comparisons: bench.py --gemv-flags)
        self._w_buf = None  # set by the engine
        self._replaced_lanes = []
        self._stale = False
        self._bind()

        # rank tables: the kernels' own (unit = 512 where rows allow it) and
        # the two the reference exposes
        self._unit = pick_unit(self.in_features)
        ready = packed.get("table512")  # left by the device encoder
        flat = ready.cuda() if ready is not None else self._dp.prefix_build(FUSED_TILE)
        self.register_buffer("_table", flat if self._unit == FUSED_TILE else self._dp.prefix_build(self._unit))
        # Rows of other lengths: whole decodes go by units of 512 all the same, counted over the row ends, which is what the
        # fast decoders take (17408 x 5088 at 55 / 40 / 5 %: 59 us, against some 300 in the general decoder).
        self.register_buffer("_flat_table", None if self._unit == FUSED_TILE else flat, persistent=False)
        self._table_ptr = self._table.data_ptr()
        if self.N % TRITON_BLOCK == 0 and TRITON_BLOCK % self._unit == 0:
            blk_table = self._table[:, :: TRITON_BLOCK // self._unit][:, : self.N // TRITON_BLOCK]
        else:
            blk_table = self._dp.prefix_build(TRITON_BLOCK)[:, :-1]
        self.register_buffer("_b1_blk", blk_table[0].contiguous())
        self.register_buffer("_b2_blk", blk_table[1].contiguous() if n_levels > 2 else torch.zeros_like(blk_table[0]))
        self._use_triton = True

        self._use_fused = True
        self._gemm_ok = True  # False: prompts are decoded and multiplied by the library
        self._gemm_fits = True
        self._split_chunk = 0
        per_row = self.in_features // self._unit
        split = _pick_split(self.in_features) if self.out_features < self.in_features else 1
        if split > 1 and self.in_features % FUSED_TILE == 0:
            self._split_chunk = self.in_features // split
            step = self._split_chunk // self._unit
        else:
            step = per_row
        q = self._table[:, : self.out_features * per_row : step]
        self.register_buffer("_q1", q[0].contiguous())
        self.register_buffer("_q2", q[1].contiguous() if n_levels > 2 else torch.zeros_like(q[0]))
        self._y32 = None

        if lanes:
            self._make_lanes()
        # the shared scratch takes its final size now, not inside some later forward (or graph capture)
        need = self._dp.gemv_workspace_bytes(self._unit, MAX_FUSED_ROWS)
        if self._lanes is not None:
            need = max(need, *(self._lanes.gemv_workspace_bytes(n) for n in range(1, MAX_FUSED_ROWS + 1)))
        shared_workspace(self._scale.device, need)

    def _make_lanes(self):
        """Lay the weights out for the lanes of the fused kernels (``_lib.LanePacked``), unless that would leave less than
        a quarter of the GPU's memory or take more than the bf16 weight: then the forwards read the packed streams.

        The layout is whole blocks of 4 rows x 512 columns.  Rows of 520 columns take 7.8 to 11.4 bits a weight and gain from
        it (16384 x 520, one token 8 us against 25), rows of 64 take 42 where bf16 takes 16 (16384 x 64, one token 7.0 us
        against 6.8, 100 rows 16 against 10)."""
        self._lanes = None
        n_bytes = _lane_bytes(self.level_bits, self.out_features, self.in_features, self.counts)
        free, total = torch.cuda.mem_get_info(self._scale.device)
        if not n_bytes or free - n_bytes - 2 * self.N < total // 4 or not _lib.LanePacked.holds(self._scale):
            for name in LANE_BUFFERS:
                self.register_buffer(name, None, persistent=False)
            self._bind()
            return
        lanes = _lib.LanePacked.build(self._dp, *self._decode_table(), self.counts)
        self._listed_quads = lanes.listed_quads
        for name, t in zip(LANE_BUFFERS, lanes.tensors):
            self.register_buffer(name, t, persistent=False)
        self._bind()

    def _fused_gemm_wins(self, rows: int) -> bool:
        """Whether ``ixh_gemm`` beats decode + library GEMM when a decode buffer is at hand.

        Only its 128-row tile kernel does (3-bit first level, at least 97 % of the elements there, more
        than 2**24 elements), and only up to 512 activation rows, beyond which it decodes the weight once
        per 512 rows.  Measured on MI355X against the tuned library GEMM, 5120 x 17408: 70 / 77 / 111 us
        against 94 / 127 / 158 us at 128 / 256 / 512 rows; 4096 x 14336: 92 / 95 / 121 against
        105 / 113 / 142; 17408 x 5120: 82 / 95 / 142 against 80 / 96 / 126, which is why layers with more
        outputs than inputs go back to the library from 257 rows on."""
        return (self.level_bits[0] == 3 and self.N > (1 << 24) and self.counts[0] * 100 >= self.N * 97
                and (rows <= 256 or (rows <= 512 and self.in_features >= self.out_features)))

    def _lanes_gemm_wins(self, rows: int) -> bool:
        """Whether the lanes' decode into matrix-core tiles (``ixh_lanes_gemm``) is the fastest way for a prompt of so many rows.

        MI355X, us from graphs, a layer without lanes (decode + library GEMM or, for tensors almost all level 1, ``ixh_gemm``)
        against this.  5 bits a weight (55 / 40 / 5 %) at 64 / 100 / 128 / 160 / 256 rows: 10240 x 5120 62 / 64 / 66 / 71 / 84
        against 27 / 35 / 37 / 49 / 57, 17408 x 5120 90 / 94 / 94 / 101 / 115 against 42 / 55 / 61 / 75 / 85.  3 bits at 64 / 100 /
        200 / 256: 10240 x 5120 65 / 66 / 70 / 70 against 28 / 35 / 49 / 49, 17408 x 5120 96 / 101 / 111 / 115 against 46 / 53 / 76
        / 77.  8 bits, which have no list, at 64 / 100 / 160: 10240 x 5120 62 / 62 / 71 against 28 / 35 / 45, 17408 x 5120 102 /
        106 / 116 against 49 / 55 / 68, 4096 x 4096 30 / 31 / 39 against 17 / 23 / 24.  From 2**24 to 3 * 2**23 weights the lanes win
        to 256 rows (at 240 / 256: 6144 x 4096, 5 bits, 41 / 53 against 34 / 35, 5120 x 4608, 3 bits, 39 / 54 against 32 / 35, 8192 x
        2560, 8 bits, 36 / 44 against 28 / 28, 24576 x 1024, 5 bits, 39 / 38 against 38 / 36; at worst, a tenth of 4 bits listed, 42
        against 43) and no further: 4096 x 4096, 5 bits, at 384 / 512 rows 37 / 41 against 36 / 42.  Below 2**24
        weights the decode, the GEMM and the host's way through both weigh more: 12000 x 768 at 256 rows 35 against 29, 2048 x 2048
        23 against 21 (eager: 31 against 20).  Up to 2**23 weights that holds to 512 rows where the list is short, one quad of listed
        elements or fewer to 50 weights (5 % of a layer's), and the rows are not so many and short that the library's product is next
        to free, at 264 / 512 rows: 2048 x 4096, 4 bits, 35 / 37 against 24 / 30, 1024 x 8192 39 / 39 against 22 / 30, 8192 x 1024,
        5 bits, 27 / 28 against 22 / 27, 2048 x 1024 15 / 17 against 12 / 15 (eager 31 / 30 against 12 / 14); with a tenth
        listed 2048 x 2048, 4 bits, 24 / 28 against 22 / 38, and 16384 x 256, 3 bits, 18 / 20 against 21 / 30.  Up to 2**20 weights it
        holds to 1024 rows whatever the list: at 640 / 1024 1024 x 1024, 5 bits, 15 / 15 against 13 / 14 (eager 32 / 31 against 12 /
        14), 512 x 2048, 4 bits, a tenth listed, 20 / 21 against 17 / 19; 1024 x 4096, 3 bits, 28 against 30 there.  Layers of at
        most 2**18 weights keep decoding into their buffer (12 us at 100 rows; the lanes took 8), which callers see there.  Rows of
        up to 256 columns: 16384 x 256 at 80 / 100 rows 17 / 17 against 13 / 15 (eager 32 / 31 against 11 / 14).

        Above 3 * 2**23 weights and 128 rows the call takes tiles of up to 512 rows, whose decode the products hide: at 192 /
        256 / 384 / 512 rows 5120 x 17408 (3 bits) 88 / 93 / 117 / 125 without lanes against 59 / 69 / 82 / 101, 10240 x 5120 (5
        bits) 80 / 84 / 81 / 92 against 52 / 56 / 66 / 84, 5120 x 5120 55 / 64 / 50 / 58 against 35 / 38 / 44 / 55.  Above 512 rows
        only layers of more than 2**26 weights gain whatever the count: 768 / 1024 rows 12288 x 6144 163 / 174 against 136 / 172,
        17408 x 5120 191 / 225 against 160 / 198, 5120 x 17408 250 / 298 against 157 / 198, 40000 x 2048 194 / 227 against 163 / 211
        (10240 x 5120 at 768 109 / 107).  Planes of 4 and 8 bits, decode + library against this, at 129 / 256 / 512 rows: 5120 x 5120
        (4 bits) 48 / 68 / 61 against 32 / 35 / 52, 17408 x 5120 (4 bits) 106 / 119 / 141 against 61 / 78 / 116, 10240 x 5120
        (8 bits) 67 / 85 / 90 against 40 / 53 / 78, 5120 x 17408 (8 bits) 199 / 249 / 217 against 56 / 72 / 105; at 1024 rows
        12288 x 6144 161 against 160 (4 bits) and 165 against 159 (8 bits)."""
        n = self.N
        if self._lanes is None or self._gemv_flags or self.in_features % 8 or n <= 1 << 18 or rows * self.in_features >= 1 << 31:
            return False
        light = n <= 1 << 23 and self.out_features <= 8192 and 50 * self._listed_quads <= n
        return rows <= 256 or (rows <= 512 and (light or n > 3 << 23)) or (rows <= 1024 and (n <= 1 << 20 or n > 1 << 26))

    def _bind(self):
        n_levels = len(self.level_bits)
        self._dp = _lib.DevicePacked(
            self.level_bits, self.out_features, self.in_features,
            [getattr(self, f"_b{i + 1}") for i in range(n_levels - 1)],
            [getattr(self, f"_l{i + 1}") for i in range(n_levels)],
            self._scale.reshape(1),
        )
        # what every fused call passes unchanged (the table follows the module when it moves: see _apply)
        import ctypes
        self._struct_ref = ctypes.byref(self._dp.struct)
        self._table_ptr = self._table.data_ptr() if hasattr(self, "_table") else None
        self._lanes = self._lane_ref = self._bias_ptr = None
        if getattr(self, LANE_BUFFERS[0], None) is not None:
            self._lanes = _lib.LanePacked(self.out_features, self.in_features, [getattr(self, b) for b in LANE_BUFFERS],
                                          self._scale)
            self._lane_ref = ctypes.byref(self._lanes.struct)
            bias = self._bias
            if bias is not None and bias.dtype is torch.bfloat16 and bias.is_cuda and bias.is_contiguous():
                self._bias_ptr = bias.data_ptr()  # added by the kernel
        self._gemv_fn = _lib.lib().ixh_lanes_gemv if self._lanes is not None else _lib.lib().ixh_gemv
        # the forward of up to MAX_FUSED_ROWS rows from the lanes, in native code
        self._native = self._native_fn = None
        if self._lanes is not None and (self._bias is None or self._bias_ptr):
            dev = self._scale.device
            self._native_fn = self._gemv_fn
            self._native = _lib.host().Forward(
                ctypes.cast(self._gemv_fn, ctypes.c_void_p).value, ctypes.addressof(self._lanes.struct), self._bias_ptr or 0,
                self.in_features, self.out_features, dev.index,
                (0,) + tuple(self._lanes.gemv_workspace_bytes(n) for n in range(1, MAX_FUSED_ROWS + 1)),
                (self._lanes, self._bias), _workspaces, dev, _lib.check,
                *(ctypes.cast(f, ctypes.c_void_p).value
                  for f in (_lib.lib().ixh_lanes_gemm, _lib.lib().ixh_lanes_gemm_workspace_bytes)))
        self._forget_plans()

    def _apply(self, fn, recurse=True):
        # .to()/.cuda() may move the buffers: point the kernel arguments at the new storage
        out = super()._apply(fn, recurse)
        if hasattr(self, "_scale") and self._scale.is_cuda:
            self._bind()
            if self._stale:
                self._follow_streams()
        return out

    def _load_from_state_dict(self, state_dict, prefix, local_metadata, strict, missing_keys, unexpected_keys, error_msgs):
        n_errors = len(error_msgs)
        super()._load_from_state_dict(state_dict, prefix, local_metadata, strict, missing_keys, unexpected_keys, error_msgs)
        if self._scale.is_cuda:  # (with assign=True the tensors are others)
            self._bind()
        # What is derived follows a whole new set of streams only: a state of other lengths (which load_state_dict goes on to
        # raise for) or a part of one leaves streams and tables that do not belong together, and no kernel may read those.
        names = ["_table"] + [f"_b{i + 1}" for i in range(len(self.level_bits) - 1)] + [f"_l{i + 1}" for i in range(len(self.level_bits))]
        if len(error_msgs) == n_errors and all(prefix + name in state_dict for name in names):
            if self._scale.is_cuda:
                self._follow_streams()
            else:  # when the layer is back on the GPU
                self._stale = True

    def _follow_streams(self):
        """Bring what is derived from the packed streams and is no part of the state dict in line with them."""
        if self._flat_table is not None:
            self._flat_table.copy_(self._dp.prefix_build(FUSED_TILE))
        if self._lanes is not None:  # a layer that was built without lanes stays without
            if _lib.LanePacked.holds(self._scale):
                self._refresh_lanes()
            else:
                self._replaced_lanes.append(self._lanes)  # (see _refresh_lanes)
                for name in LANE_BUFFERS:
                    setattr(self, name, None)
                self._bind()
        self._stale = False

    def _refresh_lanes(self):
        """Lay the weights out again, in place: a graph captured earlier serves the new ones, as it does from the packed
        streams.  Where the new list does not fit into the old one's memory the layout is replaced as a whole and the old one
        stays alive: such a graph goes on serving the old weights and has to be captured again."""
        lanes = _lib.LanePacked.build(self._dp, *self._decode_table(), self.counts, into=self._lanes)
        self._listed_quads = lanes.listed_quads
        if lanes is not self._lanes:
            self._replaced_lanes.append(self._lanes)
            for name, t in zip(LANE_BUFFERS, lanes.tensors):
                setattr(self, name, t)
            self._bind()
        else:
            self._forget_plans()

    def _set_shared_buf(self, w_buf):
        self._w_buf = w_buf
        self._forget_plans()

    def _forget_plans(self):
        self._plans = {}
        if self._native is not None:
            self._native.any_rows = self._packed_rows()  # rows up to which calls that are not plain go to the lanes too: see _fused_plan
            # (what _lanes_gemm_wins allows for a count of rows, it allows for fewer)
            self._native.many_rows = max((rows for rows in (256, 512, 1024) if self._lanes_gemm_wins(rows)), default=0)

    def _decode_table(self):
        """The rank table and unit of a decode of the whole weight."""
        return (self._table, self._unit) if self._flat_table is None else (self._flat_table, FUSED_TILE)

    def _decode(self):
        """Decode into the shared buffer and return it as ``[out_f, in_f]``
        (reference ``ixrun/engine.py:109-133``)."""
        w_flat = self._w_buf[: self.N]
        self._dp.decode(*self._decode_table(), out_bf16=w_flat)
        return w_flat.view(self.out_features, self.in_features)

    def _packed_rows(self) -> int:
        """Most rows that one call of ``ixh_gemv`` on the packed streams is the fastest way for."""
        if self._w_buf is None:
            return MAX_FUSED_ROWS
        if self.counts[0] * 100 >= self.N * 97:
            return MAX_FUSED_ROWS_WITH_BUFFER
        return MAX_FUSED_ROWS_WITH_BUFFER_DENSE if self.level_bits == (3, 5, 8) else 1

    def _fused_plan(self, rows):
        """How a forward of `rows` activation rows is served by the fused kernel: the row count of each call (one, or
        two for 17 .. 32 rows on a large layer that is almost all level 1) with the scratch it needs, or False where
        the many-row paths take over; and whether that holds for plain calls only, because without lanes the rows would go
        through decode + ``F.linear``, which serves gradients, transforms and autocast.  Worked out once per row count;
        ``_set_shared_buf`` and ``_bind`` forget the answers."""
        lanes = self._lanes is not None and self._gemv_flags == 0
        packed_rows = self._packed_rows()
        fused_rows = MAX_FUSED_ROWS if lanes else packed_rows
        two_calls = MAX_FUSED_ROWS < rows <= 2 * MAX_FUSED_ROWS and self.N >= SPLIT_FUSED_MIN_WEIGHTS
        two_packed_calls = two_calls and packed_rows == MAX_FUSED_ROWS and self.counts[0] * 100 >= self.N * 97
        two_calls = two_calls and not self._lanes_gemm_wins(rows) if lanes else two_packed_calls
        plan = False
        if 1 <= rows <= fused_rows or two_calls:
            calls = []
            for r0 in range(0, rows, MAX_FUSED_ROWS):
                n = min(MAX_FUSED_ROWS, rows - r0)
                calls.append((r0, n, self._lanes.gemv_workspace_bytes(n) if lanes
                              else self._dp.gemv_workspace_bytes(self._unit, n, self._gemv_flags)))
            plan = (lanes, tuple(calls), rows > packed_rows and not two_packed_calls)
        self._plans[rows] = plan
        return plan

    def forward(self, x):
        if self._native is not None and self._use_fused and not self._gemv_flags and self._gemv_fn is self._native_fn:
            y = self._native(x)
            if y is None and self._gemm_ok:
                y = self._native.many(x)
            if y is not None:
                return y
        if x.is_cuda and x.device.index not in (None, _current_device()):  # (the null stream is the current device's)
            with torch.cuda.device(x.device):
                return self.forward(x)
        in_f = self.in_features
        if self._use_fused and x.dtype is torch.bfloat16 and x.is_cuda and in_f and x.shape[-1] == in_f:
            rows = x.numel() // in_f
            plan = self._plans.get(rows)
            if plan is None:
                plan = self._fused_plan(rows)
            if plan and (not plan[2] or _plain_call(x)):
                # one ctypes call with the arguments that never change kept bound
                out_f = self.out_features
                if not x.is_contiguous():
                    x = x.contiguous()
                dev = x.device
                y = torch.empty(x.shape[:-1] + (out_f,), dtype=torch.bfloat16, device=dev)
                x_ptr, y_ptr = x.data_ptr(), y.data_ptr()
                stream = _raw_stream(dev.index if dev.index is not None else torch.cuda.current_device())
                lanes, calls, _ = plan
                for r0, n, ws_bytes in calls:  # one call, or two on the same stream and workspace
                    ws = _workspaces.get(dev) if ws_bytes else None
                    if ws_bytes and (ws is None or ws.numel() * 4 < ws_bytes):
                        ws = shared_workspace(dev, ws_bytes)
                    if lanes:
                        rc = self._gemv_fn(self._lane_ref, x_ptr + r0 * in_f * 2, in_f, self._bias_ptr, n, y_ptr + r0 * out_f * 2,
                                           out_f, ws.data_ptr() if ws_bytes else None, ws_bytes, stream)
                    else:
                        gemv = self._gemv_fn if self._lanes is None else _lib.lib().ixh_gemv
                        rc = gemv(self._struct_ref, self._table_ptr, self._unit, x_ptr + r0 * in_f * 2, n, in_f,
                                  y_ptr + r0 * out_f * 2, out_f, None, ws.data_ptr() if ws_bytes else None,
                                  ws_bytes, self._gemv_flags, stream)
                    if rc:
                        _lib.check(rc)
                if self._bias is not None and not (lanes and self._bias_ptr):
                    y = y + self._bias.to(y.dtype)
                return y
        rows = x.numel() // in_f if in_f else 0
        if (self._use_fused and self._gemm_ok and rows > MAX_FUSED_ROWS and x.dtype is torch.bfloat16 and x.is_cuda and x.shape[-1] == in_f
                and self._lanes_gemm_wins(rows) and x.device == self._scale.device and _plain_call(x)):
            x2 = x.reshape(rows, in_f).contiguous()
            if x2.data_ptr() % 16:
                x2 = x2.clone()
            y = torch.empty((rows, self.out_features), dtype=torch.bfloat16, device=x.device)
            try:
                self._lanes.gemm(x2, y, self._bias if self._bias_ptr else None)
            except torch.OutOfMemoryError:
                if self._w_buf is None:
                    raise
                # no room for the slices' sums (128 MiB and the activations at most): the decode buffer is there already
                del x2, y
                return self._decode_and_multiply(x)
            if self._bias is not None and not self._bias_ptr:
                y = y + self._bias.to(y.dtype)
            return y.view(x.shape[:-1] + (self.out_features,))
        if (self._use_fused and self._gemm_ok and self._gemm_fits and x.dtype == torch.bfloat16 and x.is_cuda and rows > MAX_FUSED_ROWS
                and x.shape[-1] == self.in_features and self._unit == 512
                and (self._w_buf is None or self._fused_gemm_wins(rows))):
            # many rows: decode tiles on chip straight into the matrix-core GEMM, no bf16 weight in HBM
            x2 = x.reshape(rows, self.in_features)
            if x2.stride(1) != 1:
                x2 = x2.contiguous()
            y = torch.empty((rows, self.out_features), dtype=torch.bfloat16, device=x.device)
            ws = shared_workspace(x.device, self._dp.gemm_workspace_bytes(rows))
            try:
                self._dp.gemm(self._table, x2, y, ws)
            except _lib.IxhError as e:
                if e.code != _lib.IXH_EUNSUPPORTED:
                    raise
                self._gemm_fits = False  # shape the fused GEMM does not take: decode + GEMM from here on
            else:
                y = y.view(x.shape[:-1] + (self.out_features,))
                if self._bias is not None:
                    y = y + self._bias.to(y.dtype)
                return y
        return self._decode_and_multiply(x)

    def _decode_and_multiply(self, x):
        w = self._decode()
        bias = self._bias.to(x.dtype) if self._bias is not None else None
        return gemm_tuning.linear(x, w.to(x.dtype) if w.dtype != x.dtype else w, bias)


class GraphLinear(nn.Module):
    """GEMM-only layer whose weight buffer is refreshed by a captured graph of
    decode launches (reference ``ixrun/engine.py:179-196``)."""

    def __init__(self, packed: dict, bias=None, decode_buf=None):
        super().__init__()
        self.out_features = packed["out_f"]
        self.in_features = packed["in_f"]
        self.N = packed["N"]
        self._w_buf = decode_buf
        if bias is not None:
            self.register_buffer("_bias", bias.detach().clone().cuda())
        else:
            self._bias = None

    def forward(self, x):
        w = self._w_buf[: self.N].view(self.out_features, self.in_features)
        bias = self._bias.to(x.dtype) if self._bias is not None else None
        return gemm_tuning.linear(x, w, bias)


class ResourceScheduler:
    """Memory estimates and a mode recommendation (reference ``ixrun/engine.py:202-235``).

    A streaming deploy keeps ``packed_storage_MB``, ``lane_storage_MB`` (the layout that the forwards read; nothing with
    ``lanes=False``) and ``shared_decode_buf_MB`` on the GPU.  With lanes a prompt takes memory for its call besides: its
    activations once more and, from 129 rows on large layers, up to 128 MiB of sums (less below); where there is no room for
    them it goes through the decode buffer."""

    @staticmethod
    @torch.no_grad()
    def estimate(model: nn.Module, level_bits=(3, 5, 8)) -> dict:
        bf16_bytes = packed_bytes = lane_bytes = n_elems = max_layer = 0
        for _, mod in iter_quantizable_linears(model):
            w = mod.weight.data
            packed = int8x_quantize(w, level_bits)
            packed_bytes += packed["total_bytes"]
            lane_bytes += _lane_bytes(packed["level_bits"], packed["out_f"], packed["in_f"], packed["counts"])
            bf16_bytes += w.numel() * 2
            n_elems += w.numel()
            max_layer = max(max_layer, w.numel())
        return {
            "bf16_weight_MB": bf16_bytes / 1e6,
            "packed_storage_MB": packed_bytes / 1e6,
            "lane_storage_MB": lane_bytes / 1e6,
            "compression": bf16_bytes / max(packed_bytes, 1),
            "max_layer_elems": max_layer,
            "shared_decode_buf_MB": max_layer * 2 / 1e6,
            "n_elems": n_elems,
        }

    @staticmethod
    def recommend(model: nn.Module, gpu_budget_GB: float, level_bits=(3, 5, 8)) -> str:
        est = ResourceScheduler.estimate(model, level_bits)
        return "cached" if est["bf16_weight_MB"] + 1500 <= gpu_budget_GB * 1000 else "streaming"


class Int8XEngine:
    """Load a model, deploy it on packed weights, generate.

    Same construction and deploy modes as the reference's ``Int8XEngine``
    (``ixrun/engine.py:241-516``).  The three ``_deploy_*`` helpers take any
    ``nn.Module``; ``from_pretrained`` needs ``transformers`` and a local
    checkpoint, as in the reference.
    """

    def __init__(self, model, tokenizer, stats=None, graph_replay=None):
        self.model = model
        self.tokenizer = tokenizer
        self.stats = stats or {}
        self._graph_replay = graph_replay
        self.model.eval()

    @classmethod
    def from_pretrained(cls, model_path: str, mode: str = "cached", level_bits=(3, 5, 8),
                        dtype=torch.bfloat16, verbose: bool = True, cache_path: str | None = None, lanes: bool = True):
        from transformers import AutoModelForCausalLM, AutoTokenizer

        tokenizer = AutoTokenizer.from_pretrained(model_path, trust_remote_code=True)
        if tokenizer.pad_token is None:
            tokenizer.pad_token = tokenizer.eos_token
        big = mode in ("streaming", "graph")
        model = AutoModelForCausalLM.from_pretrained(model_path, dtype=dtype, low_cpu_mem_usage=True)
        if not big:
            model = model.cuda()
        if mode == "streaming":
            stats = cls._deploy_streaming(model, level_bits, verbose=verbose, cache_path=cache_path, lanes=lanes)
        elif mode == "graph":
            stats, replay = cls._deploy_graph(model, level_bits, verbose=verbose)
            return cls(model, tokenizer, stats, graph_replay=replay)
        else:
            stats = cls._deploy_cached(model, level_bits, verbose=verbose)
        eng = cls(model, tokenizer, stats)
        if big:
            eng._finalize_device()
        return eng

    # ----- deploy helpers ---------------------------------------------------
    @staticmethod
    def _deploy_cached(model, level_bits, verbose=True):
        from .linear import deploy_model

        return deploy_model(model, level_bits=level_bits, cache="full", verbose=verbose)

    @staticmethod
    @torch.no_grad()
    def _deploy_streaming(model, level_bits, verbose=True, cache_path=None, lanes=True):
        """Packed weights resident on the GPU plus one shared decode buffer
        (reference ``ixrun/engine.py:343-416``).  ``cache_path`` names a file of
        already packed layers, ``{"level_bits": ..., "layers": [(name, packed,
        bias), ...]}``, written on the first deploy and read on later ones; a
        cache built with other ``level_bits`` or for other layer names raises
        ``ValueError`` as in the reference (``:360-370``).

        With ``lanes`` every layer also keeps the lane layout that its forwards read, while a quarter of the GPU's memory
        stays free: the layers deployed last may go without and are slower for it.  The statistics say how many have one
        (``n_lane_layers``), its bytes (``lane_bytes``) and all that the layers hold on the GPU (``resident_bytes``: packed
        streams, rank tables, lanes, biases); ``total_bytes`` are the packed streams, as in the reference."""
        targets = list(iter_quantizable_linears(model))
        layer_data = None
        if cache_path is not None and os.path.exists(cache_path):
            if verbose:
                print(f"[engine][cache] loading packed weights from {cache_path}", flush=True)
            # tuples, dicts, numbers and tensors only: the safe loader reads all of it
            blob = torch.load(cache_path, map_location="cpu", weights_only=True)
            if tuple(blob["level_bits"]) != tuple(level_bits):
                raise ValueError(
                    f"cache was built with level_bits={blob['level_bits']}, "
                    f"requested {tuple(level_bits)}; delete the cache or change level_bits")
            layer_data = blob["layers"]
            have = {n for n, _ in model.named_modules()}
            missing = [n for n, _, _ in layer_data if n not in have]
            if missing:
                raise ValueError(f"cache/model mismatch: {len(missing)} unknown layers")
            if verbose:
                print(f"[engine][cache] {len(layer_data)} layers loaded", flush=True)
        if layer_data is None:
            layer_data = []
            for name, mod in targets:
                bias = mod.bias.data if mod.bias is not None else None
                layer_data.append((name, quantize_for_deploy(mod.weight.data, level_bits), bias))
            if cache_path is not None:
                if verbose:
                    print(f"[engine][cache] saving packed weights to {cache_path}", flush=True)
                torch.save({"level_bits": tuple(level_bits),
                            "layers": [(n, portable_packed(p), b) for n, p, b in layer_data]}, cache_path)

        total_bytes = max_n = 0
        layers = []
        for name, packed, bias in layer_data:
            layers.append((name, StreamingLinear(packed, bias=bias, lanes=lanes)))
            total_bytes += packed["total_bytes"]
            max_n = max(max_n, packed["N"])
        shared_w = torch.empty(max_n, dtype=torch.bfloat16, device="cuda")
        for name, sl in layers:
            sl._set_shared_buf(shared_w)
            _set_parent_child(model, name, sl)
        gc.collect()
        torch.cuda.empty_cache()
        shared_mb = shared_w.numel() * 2 / 1e6
        laid_out = [sl._lanes.nbytes for _, sl in layers if sl._lanes is not None]
        resident = sum(b.numel() * b.element_size() for _, sl in layers for b in sl.buffers())
        if verbose:
            print(f"[engine][streaming] {len(layers)} layers | packed={total_bytes / 1e6:.0f}MB | "
                  f"lane layout={sum(laid_out) / 1e6:.0f}MB on {len(laid_out)} layers | GPU-resident={resident / 1e6:.0f}MB | "
                  f"shared decode buf={shared_mb:.1f}MB", flush=True)
        return {"mode": "streaming", "n_layers": len(layers), "total_bytes": total_bytes, "shared_gpu_MB": shared_mb,
                "lane_bytes": sum(laid_out), "n_lane_layers": len(laid_out), "resident_bytes": resident}

    @staticmethod
    @torch.no_grad()
    def _deploy_graph(model, level_bits, verbose=True):
        """Streaming deploy with every layer's decode launch captured in one
        graph (reference ``ixrun/engine.py:420-487``): each layer gets its own
        decode buffer, the graph replays all decodes, forwards are GEMM-only."""
        targets = list(iter_quantizable_linears(model))
        total_params = sum(m.weight.numel() for _, m in targets)
        if total_params * 2 > torch.cuda.get_device_properties(0).total_memory * 0.9:
            raise RuntimeError(
                f"graph mode needs {total_params * 2 / 1e9:.1f}GB of per-layer decode buffers "
                f"- too large for this GPU; use mode='streaming'")
        total_bytes = 0
        specs = []
        for name, mod in targets:
            packed = quantize_for_deploy(mod.weight.data, level_bits)
            bias = mod.bias.data if mod.bias is not None else None
            sl = StreamingLinear(packed, bias=bias, lanes=False)  # only its decode is used
            buf = torch.empty(packed["N"], dtype=torch.bfloat16, device="cuda")
            sl._set_shared_buf(buf)
            specs.append((name, sl, buf))
            total_bytes += packed["total_bytes"]

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _, sl, _ in specs:
                sl._decode()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _, sl, _ in specs:
                sl._decode()
        torch.cuda.synchronize()
        if verbose:
            print(f"[engine][graph] captured {len(specs)} decode kernels", flush=True)
        for name, sl, buf in specs:
            meta = {"out_f": sl.out_features, "in_f": sl.in_features, "N": sl.N}
            _set_parent_child(model, name, GraphLinear(meta, bias=sl._bias, decode_buf=buf))

        def replay(_keep_alive=specs, _graph=graph):
            _graph.replay()

        if verbose:
            print(f"[engine][graph] {len(specs)} layers | packed={total_bytes / 1e6:.0f}MB | decode=graph.replay()",
                  flush=True)
        return {"mode": "graph", "n_layers": len(specs), "total_bytes": total_bytes}, replay

    # ----- inference --------------------------------------------------------
    def _finalize_device(self):
        """Move whatever the deploy left on the CPU (reference ``ixrun/engine.py:490-504``)."""
        for _, mod in self.model.named_modules():
            for p in mod.parameters(recurse=False):
                if p.data.device.type != "cuda":
                    p.data = p.data.cuda()
            for bname, b in mod.named_buffers(recurse=False):
                if b.device.type != "cuda":
                    setattr(mod, bname, b.cuda())
        gc.collect()
        torch.cuda.empty_cache()
        self.model.eval()

    def _pre_forward(self):
        if self._graph_replay is not None:
            self._graph_replay()

    @torch.no_grad()
    def generate(self, prompt, max_new_tokens: int = 64, **kw):
        """Greedy text generation through the wrapped model's own ``generate``."""
        self._pre_forward()
        ids = self.tokenizer(prompt, return_tensors="pt").to("cuda")
        out = self.model.generate(**ids, max_new_tokens=max_new_tokens, do_sample=False, **kw)
        return self.tokenizer.decode(out[0][ids["input_ids"].shape[1]:], skip_special_tokens=True)
