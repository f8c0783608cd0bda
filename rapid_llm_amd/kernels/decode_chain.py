"""All layers of a recorded decode step of few tokens in one launch (csrc/decode_chain.hip).

The layers are the dense decoder's (rapid_llm/models/base.py:231-266: norm, packed q | k | v product, attention,
output product, norm, gate and up, down); the launch computes what their own kernels would, with the same
rounding of everything that is stored."""

from __future__ import annotations

import ctypes
from typing import Optional, Sequence

import torch

from . import build
from .ops import KernelError, _need, _ok, _p, _stream, chip

HEAD_DIM = 128
MAX_ROWS = 16
MAX_GROUP = 4  # query heads a kv head
TAGGED_ROWS = 2  # rows up to which results travel with the launch's number
MIN_KEYS = 256  # keys that a share of a request's context has at least
MAX_SHARES = 16  # of a request's keys: whoever folds them asks for all
STEP = 128  # every contraction is a multiple of it
# Rows of a recorded step up to which: keys of its longest context up to which, and a layer's matrix elements (in units of 2^20) up to
# which, the launch is the faster one.  What it saves are the starts and tails of six kernels a layer; what it costs is that a phase's
# last workgroups leave the memory idle where weights, or the keys of many requests, keep it busy.  Time of the launch over that of
# the layers' own kernels, 28 layers of 15.7 / 19.7 / 23.2 / 28.3 / 38.5 / 50.3 / 56.8 / 63.7 M elements (the first and the sixth
# are Qwen3-0.6B's and 1.7B's; the dividing lines lie between a size below 1 and one above, 1.7B's own two rows and 2 to 8 of
# 28 M among them):
#   1 row, 300 keys 0.82 / 0.89 / 0.91 / 0.92 / 0.99 / 0.95 / 1.04 / 1.05, 8,000 0.90 / 0.93 / . / . / . / 0.98, 16,000 0.99 / 1.01,
#   32,000 1.05; 2 rows, 42 to 546 keys 0.83 / 0.99 / 0.93 / 1.04 / 1.05 / 1.03 / . / 1.04, 2,000 to 4,000 0.92 / 1.00 / . / 1.06, 8,000 0.94 / 1.00,
#   500 to 16,000 0.95 / 1.03; 4 rows, 64 to 900 0.91 / 1.00 / 1.05 / 1.05 / 1.04 / 1.00 / . / 1.08, 200 to 4,000 0.97 / 1.00 / . / 1.04, 8,000 0.97 / 1.02,
#   500 to 16,000 0.99 / 1.05; 8 rows, 64 to 900 0.87 / 0.99 / 1.04 / 1.02 / 1.04 / 1.00 / . / 1.04, 1,000 to 2,000 0.93 / 0.96, 200 to 4,000 1.02 / 1.02;
#   12 rows, 64 to 900 . / 0.99 / 0.99 / 0.99 / 1.03 / 1.01 / 1.07 / 1.05, 1,000 to 2,000 0.98 / 1.04, 200 to 4,000 1.10 / 1.16; 16 rows, 64 to 900
#   0.87 / 0.95 / 0.93 / 0.93 / 0.97 / 0.96 / 0.97 / 0.98 (76.0 M: 1.02), 200 to 2,000 0.96 / 0.99 / . / 0.99 / 1.01 / 0.99, 200 to 4,000 1.01 / 1.04 / . / 1.03 / 1.04 / 1.01.
_FASTER = {
    1: ((8192, 50), (16384, 16)),
    2: ((1024, 24), (4096, 20), (16384, 16)),
    4: ((4096, 20), (16384, 16)),
    8: ((2048, 20),),
    15: ((1024, 32), (2048, 16)),
    16: ((2048, 64),),
}

_lib: ctypes.CDLL | None = None


def _library() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        lib = build.load(build.decode_chain_library())
        limits = (lib.rl_decode_chain_max_group(), lib.rl_decode_chain_min_keys())
        if limits != (MAX_GROUP, MIN_KEYS):
            raise KernelError(f"the decode chain's limits {limits} are not the launch rules'")
        lib.rl_decode_chain_space.restype = lib.rl_decode_chain_shares.restype = ctypes.c_longlong
        lib.rl_decode_chain_last_launch.restype = ctypes.c_uint
        _lib = lib
    return _lib


def faster(rows: int, weights: int, span: int) -> bool:
    """Whether the launch is the faster one for ``rows`` rows over layers of ``weights`` matrix elements and contexts of up to ``span`` keys."""
    limits = next(limits for most, limits in _FASTER.items() if rows <= most)
    return weights <= next((limit << 20 for keys, limit in limits if span <= keys), 0)


def fits(rows: int, hidden: int, nq: int, nkv: int, d: int, inter: int, page_size: int, span: int = 1) -> bool:
    """Whether the launch takes layers of these sizes, and is the faster one over contexts of up to ``span`` keys."""
    return (
        1 <= rows <= MAX_ROWS and d == HEAD_DIM and nkv >= 1 and nq % nkv == 0 and nq // nkv <= MAX_GROUP
        and hidden % STEP == 0 and inter % STEP == 0 and page_size % 8 == 0
        and faster(rows, hidden * ((2 * nq + 2 * nkv) * d + 3 * inter), span)
    )


def shares(rows: int, nkv: int, span: int, units: int | None = None) -> int:
    """Shares that a request's keys are dealt to at most: a workgroup's worth of keys on every compute unit, as far
    as there are keys for it."""
    units = chip().units if units is None else units
    return max(1, min(-(-span // MIN_KEYS), units // (rows * nkv), MAX_SHARES))


def takes(layers: int, rows: int, hidden: int, nq: int, nkv: int, inter: int, columns: int, page_size: int, span: int) -> bool:
    """Whether the launch's index arithmetic reaches so many layers and so large a cache (``columns`` of the block table)."""
    return bool(_library().rl_decode_chain_takes(layers, rows, hidden, nq, nkv, inter, columns, page_size, shares(rows, nkv, span), chip().units))


class Space:
    """What the launches of a model's recorded steps share: rows between the products, shares of the attention, and
    what the workgroups of a launch know of each other.  One launch uses it at a time (a runner's steps follow each other)."""

    def __init__(self, layers: int, hidden: int, nq: int, nkv: int, inter: int, span: int, device) -> None:
        sizes = space_bytes(layers, hidden, nq, nkv, inter, span)
        # (what lies in the place of a launch's number must be an earlier launch's)
        self.tagged, self.rows, self.shares, self.control = (torch.zeros(n, dtype=torch.uint8, device=device) for n in sizes)
        # a launch that is given up leaves a word in host memory, which costs nothing to look at
        self._notice = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        self._seen = self._notice.numpy()
        self.notice = ctypes.c_void_p()
        _ok(_library().rl_decode_chain_notice(_p(self._notice), ctypes.byref(self.notice)), "rl_decode_chain_notice")

    def given_up(self) -> bool:
        """Whether a launch that has ended was given up: its result, and that of every later one, is NaN."""
        return bool(self._seen[0])


def space_bytes(layers: int, hidden: int, nq: int, nkv: int, inter: int, span: int) -> tuple[int, int, int, int]:
    """Bytes of the four tensors of :class:`Space` for steps of up to ``MAX_ROWS`` rows over at most ``span`` keys."""
    lib = _library()
    return (
        lib.rl_decode_chain_space(layers, TAGGED_ROWS, hidden, nq, nkv, inter),
        lib.rl_decode_chain_space(layers, MAX_ROWS, hidden, nq, nkv, inter),
        max(lib.rl_decode_chain_shares(layers, rows, nq, shares(rows, nkv, span)) for rows in range(1, MAX_ROWS + 1)),
        lib.rl_decode_chain_control(),
    )


class DecodeChain:
    """The launch of one recorded step: its layers' table, kept as long as the graph that holds it."""

    def __init__(self, layers: Sequence[Sequence[Optional[torch.Tensor]]], space: Space, rows: int, hidden: int,
                 nq: int, nkv: int, inter: int, span: int, scale: float, eps: tuple[float, float, float]) -> None:
        """``layers``: for each the matrices (q | k | v, output, gate | up, down), the weights of the query and key norms
        (or ``None``), of the norm in front of gate and up and of the next layer's first norm (``None``: the last
        layer), and the pages of keys and values.  ``eps``: of the query and key norms, of a layer's first norm, of its
        second."""
        lib = _library()
        self.rows, self.hidden, self.nq, self.nkv, self.inter = rows, hidden, nq, nkv, inter
        self.scale, self.eps = float(scale), tuple(float(e) for e in eps)
        self.nsplit = shares(rows, nkv, span)
        self.num_layers = len(layers)
        self.page_size = layers[0][8].shape[2]
        d = HEAD_DIM
        if not fits(rows, hidden, nq, nkv, d, inter, self.page_size, span):
            raise KernelError(f"the decode chain does not take {rows} rows of layers of {hidden} / {nq} / {nkv} / {inter}")
        shapes = (((nq + 2 * nkv) * d, hidden), (hidden, nq * d), (2 * inter, hidden), (hidden, inter))
        pages = layers[0][8].shape[0]
        for i, layer in enumerate(layers):
            for w, shape in zip(layer[:4], shapes):
                _need(w, "a layer's matrix", torch.bfloat16, shape)
            for w, size in zip(layer[4:8], (d, d, hidden, hidden)):
                if w is not None:
                    _need(w, "a norm's weight", torch.float32, (size,))
            if layer[6] is None or (layer[7] is None) != (i == len(layers) - 1) or (layer[4] is None) != (layer[5] is None):
                raise KernelError("every layer of a decode chain but the last has a norm behind it")
            _need(layer[8], "key pages", torch.bfloat16, (pages, nkv, self.page_size, d))
            _need(layer[9], "value pages", torch.bfloat16, (pages, nkv, d, self.page_size))
            if any(t is not None and t.data_ptr() % 16 for t in layer):
                raise KernelError("the tensors of a decode chain begin at multiples of 16 bytes")
        if lib.rl_decode_chain_layer_bytes() != 8 * len(layers[0]):
            raise KernelError("the decode chain's table of layers is laid out otherwise")
        rows_space = space.tagged if rows <= TAGGED_ROWS else space.rows
        if (rows_space.numel() < lib.rl_decode_chain_space(self.num_layers, rows, hidden, nq, nkv, inter)
                or space.shares.numel() < lib.rl_decode_chain_shares(self.num_layers, rows, nq, self.nsplit)):
            raise KernelError("the decode chain's space is too small")
        self.space = space
        self.tensors = layers  # what the table points at
        self.table = torch.tensor([[0 if t is None else t.data_ptr() for t in layer] for layer in layers],
                                  dtype=torch.int64, device=space.control.device)

    def run(self, x: torch.Tensor, residual: torch.Tensor, positions: torch.Tensor, token_slot: torch.Tensor,
            block_table: torch.Tensor, cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], max_position: int) -> torch.Tensor:
        """The last layer's down projection (not yet in the stream) of the first norm's rows ``x``; everything before
        it is added to ``residual`` in place, and the tokens' keys and values are in their pages."""
        rows, hidden, d = self.rows, self.hidden, HEAD_DIM
        _need(x, "x", torch.bfloat16, (rows, hidden))
        _need(residual, "residual", torch.float32, (rows, hidden))
        _need(positions, "positions", torch.int32, (rows,))
        _need(token_slot, "token slots", torch.int32, (rows,))
        _need(block_table, "block_table", torch.int32)
        if (x.data_ptr() | residual.data_ptr()) % 16:
            raise KernelError("the rows of a decode chain begin at multiples of 16 bytes")
        if max_position // self.page_size >= block_table.shape[1]:
            raise KernelError(
                f"position {max_position} needs page {max_position // self.page_size} of a block table with "
                f"{block_table.shape[1]} columns"
            )
        if cos is not None:
            _need(cos, "cos table", torch.float32, (None, d // 2))
            _need(sin, "sin table", torch.float32, tuple(cos.shape))
            if max_position >= cos.shape[0]:
                raise KernelError(f"position {max_position} is beyond the rotation table of {cos.shape[0]} positions")
        out = torch.empty((rows, hidden), dtype=torch.bfloat16, device=x.device)
        _ok(
            _library().rl_decode_chain(
                _p(self.table), _p(x), _p(residual), _p(out), _p(positions), _p(token_slot), _p(block_table), _p(cos), _p(sin),
                _p(self.space.tagged), ctypes.c_longlong(self.space.tagged.numel()), _p(self.space.rows),
                _p(self.space.shares), ctypes.c_longlong(self.space.shares.numel()), _p(self.space.control), self.space.notice, self.num_layers, rows, hidden, self.nq, self.nkv, self.inter,
                block_table.stride(0), self.page_size, self.nsplit, ctypes.c_float(self.scale),
                *(ctypes.c_float(e) for e in self.eps), chip().units, _stream(),
            ),
            "rl_decode_chain",
        )
        return out
