"""Python face of the kernels in ``csrc/tile_gemm.hip``, ``pair_gemm.hip`` and ``wide_gemm.hip``: products of many rows on the matrix cores, and the rules by
which a product goes there, how it is cut into tiles and shares, and where the library's product stays."""
from __future__ import annotations

import ctypes
import functools
import math
from typing import Optional, Tuple

import torch

from ..csrc import build as _build
from . import GATED_ACTIVATIONS, SKINNY_MAX_ROWS, KernelError, _check, _gpu, _load, _off_vectors, _ptr, _stream, add_rmsnorm, core, dtype_code, rope_kv_write

COMPUTE_UNITS = 256

# Tiles of the float32 product: rows of x, rows of W, workgroups a compute unit holds, and the microseconds that 16
# elements of K take a workgroup when every unit is full and when it is alone (the matrix cores lower their clock under
# load).  Fitted to sweeps of 65 to 2,048 rows over the layer sizes of the 1B, 3B and 8B shapes, where the plan that
# :func:`split_plan` takes is within 4 % of the best of all tiles and shares.
SPLIT_TILES = ((64, 256, 2, 1.67, 0.76), (128, 128, 2, 1.48, 0.66), (128, 256, 1, 1.36, 0.88), (256, 256, 1, 2.38, 1.64))


def tile_lib() -> ctypes.CDLL:
    return _load(_build.TILE_GEMM)


def _split_cost(M: int, N: int, K: int, tile: int, shares: int, groups: int = 1) -> float:
    """Microseconds of a float32 product with this tile and this many shares, by the figures above; the kernel that adds
    the shares moves them at 4 TB/s.  ``groups``: M rows in all, of which a group's last tile is half empty."""
    bm, bn, held, loaded, alone = SPLIT_TILES[tile]
    tiles = -(-M // bm) if groups == 1 else M // bm + (groups + 1) // 2
    full, rest = divmod(tiles * -(-N // bn) * shares, COMPUTE_UNITS * held)
    steps = -(-K // (16 * shares))
    cost = 7.0 + full * loaded * steps + (alone + (loaded - alone) * rest / (COMPUTE_UNITS * held)) * steps * (rest > 0)
    return cost + (3.5 + (shares + 1) * M * N * 4 / 4e6 if shares > 1 else 0.0)


def _whole(M: int) -> int:
    """M rounded up to whole tiles of the fewest rows.  A plan is made for so many and kept: a server's steps have a new
    number of rows most of the time, and weighing all tiles and shares costs the host 10 to 60 us, more than the launch
    (a bfloat16 product of rows not seen before 24 us, of others 9.5; the library's 78 and 18)."""
    return -(-M // 64) * 64


def split_plan(M: int, N: int, K: int, gated: bool = False) -> Tuple[int, int, float]:
    """(tile, shares, estimated microseconds).  ``gated``: the product whose epilogue makes gate and up one output, which
    is not cut along K."""
    return _split_plan(_whole(M), N, K, gated)


@functools.lru_cache(maxsize=4096)
def _split_plan(M: int, N: int, K: int, gated: bool) -> Tuple[int, int, float]:
    cost, tile, shares = min((_split_cost(M, N, K, t, s), t, s) for t in range(len(SPLIT_TILES))
                             for s in ((1,) if gated else range(1, 17)) if s == 1 or K // s >= 128)
    return tile, shares, cost


def split_wins(x: torch.Tensor, rows: torch.Tensor) -> bool:
    """Whether ``x . rows^T`` goes to the float32 product of :func:`split_gemm`: more rows than the skinny product takes
    and work enough to pay for its start (some 8 us from the first load to the first matrix instruction).  Measured in
    recorded launches, each with another W, against the library's float32 product (us, library : this): 512 rows on
    [16384, 2048] 259 : 172, on [2048, 8192] 135 : 99, on [3072, 2048] 61 : 48, on [2048, 2048] 38 : 37; 164 rows on [3072, 3072]
    42 : 39, on [3072, 2048] 28 : 32, on [2048, 2048] 21 : 27; 256 rows on [3072, 2048] 40 : 34, on [2048, 2048] 22.5 : 28: the line
    lies at 2.2 GFLOP."""
    M, K = x.shape
    return (x.dtype == torch.float32 and M > 64 and K % 4 == 0 and 2.0 * M * rows.shape[0] * K >= 2.2e9 and x.is_contiguous()
            and rows.is_contiguous() and x.data_ptr() % 16 == 0 and rows.data_ptr() % 16 == 0)


def split_gemm(x: torch.Tensor, rows: torch.Tensor, out: Optional[torch.Tensor] = None, gated: Optional[str] = None, squared: bool = False,
               plan: Optional[Tuple[int, int]] = None, addends: bool = False) -> torch.Tensor:
    """``x . rows^T`` for float32 ``x`` [M, K] and ``rows`` [N, K] by six bfloat16 products of the operands' three parts
    (against 64 bits 0.6 to 0.9 times the error of the library's float32 product for sums of 700 to 8,192 numbers).  ``gated``: an activation's
    name; ``rows`` is [gate; up] stacked and the result ``act(gate) * up`` [M, N / 2].  ``squared``: ``relu(.)^2``.
    ``plan``: another (tile, shares) than :func:`split_plan`'s.  ``addends`` (without ``out`` and activations): where the product is
    cut along K its shares come back as they are, [shares, M, N], for a norm that adds them."""
    M, K = x.shape
    N = rows.shape[0]
    _gpu(x, "x", torch.float32)
    _gpu(rows, "w", torch.float32, (N, K))
    if gated is not None and (N % 2 or squared):
        raise KernelError("a gated product takes a stacked matrix and no other activation")
    _addends_alone(addends, out, gated, squared)
    cols = N if gated is None else N // 2
    if K % 4 or x.data_ptr() % 16 or rows.data_ptr() % 16:
        raise KernelError(f"rows of {K} float32 elements at this address are not aligned to 16 bytes")
    tile, shares = plan or split_plan(M, N, K, gated is not None)[:2]
    per = -(-K // (16 * shares)) * 16
    shares = -(-K // per)                                   # no share is empty
    if shares > 1:
        parts = torch.empty(shares, M, N, dtype=torch.float32, device=x.device)
    elif out is None:
        out = torch.empty(M, cols, dtype=torch.float32, device=x.device)
    if out is not None:
        _gpu(out, "out", torch.float32, (M, cols))
    _check(tile_lib().ni_split_gemm(_ptr(x), _ptr(rows), _ptr(parts if shares > 1 else out), M, N, K, tile, shares, per, int(gated is not None),
                                    GATED_ACTIVATIONS[gated or "silu"], int(squared and shares == 1), _stream()), "split_gemm")
    if shares > 1:
        return parts if addends else _add_shares(parts, torch.float32, out, squared)
    return out


def _addends_alone(addends: bool, out: Optional[torch.Tensor], gated: Optional[str], squared: bool) -> None:
    if addends and (out is not None or gated is not None or squared):
        raise KernelError("a product that leaves its addends has no out and no activation")


def _add_shares(parts: torch.Tensor, dtype: torch.dtype, out: Optional[torch.Tensor], squared: bool) -> torch.Tensor:
    """The shares [S, M, N] of a product added in their order, in ``out`` or a new tensor of that type."""
    S, M, N = parts.shape
    if out is None:
        out = torch.empty(M, N, dtype=dtype, device=parts.device)
    _check(tile_lib().ni_add_shares(_ptr(parts), _ptr(out), ctypes.c_size_t(M * N), S, int(squared), dtype_code(dtype), _stream()), "add_shares")
    return out


# ---------------------------------------------------------------- float32 by three products in half precision

# Tiles of the product in half precision: rows of x, rows of W, workgroups a compute unit holds, and in microseconds: what a
# launch takes beside its steps, 16 columns of K with one workgroup alone on its unit and with all units full, and how late between the
# two the time rises (the power of the share of the units that is taken).  Fitted to sweeps of all tiles and shares at 96 to
# 2,048 rows over the layer sizes of the 1B, 3B and 8B shapes, on two cards, recorded, every launch with another W: of 162 plans taken by time alone the
# average is 1 % above the best and the worst 12.
PAIR_TILES = ((128, 256, 1, 10.8, 0.401, 0.562, 4.48), (64, 256, 1, 9.9, 0.276, 0.330, 6.72), (128, 128, 1, 10.9, 0.219, 0.309, 4.98),
              (64, 128, 2, 9.4, 0.084, 0.437, 1.59))
PAIR_SUMS = (1, 2, 2, 2)        # sums that a share's large products are added in (SUMS of the kernel)
# The same figures of a layout with one sum a share, W in registers and 32 x 32 products.  Its plans say how many partial sums a result is made of
# at least: the fewer there are the longer each is, and every addition is rounded.  Rms error beside the rows' norms, with that layout's
# plan : by time alone : with as many sums (1e-7): 700 rows on [2048, 2048] 1.71 : 2.21 : 1.71, 1,300 on
# [2048, 8192] 3.43 : 4.15 : 2.53, 2,048 on [5120, 3072] 2.22 : 2.64 : 2.22, 600 on [16384, 3072] 2.22 : 2.64 : 2.22, 448 on [6144, 4096] 2.51 : 3.00 :
# 1.91; of 54 products and 18 with SwiGLU none is above the first by more than 0.2 %.  One plan in 70 is another by this: with the norm behind it that
# adds the shares 1 to 5 % slower (us, by time alone : so: 700 rows on [2048, 2048] 31.0 : 31.5, 2,000 on [5120, 3072] 222 : 234, 400 on [6144, 4096] 86.6 : 90.1), where a
# kernel has to add them up to 24 % (1,000 on [1536, 1536] 18.9 : 23.5, 700 on [2048, 2048] 23.6 : 27.2).
PAIR_SUM_TILES = ((128, 256, 1, 16.1, 0.447, 0.651, 4.2), (64, 256, 2, 12.4, 0.228, 0.729, 1.18), (128, 128, 2, 11.8, 0.278, 0.745, 1.25),
                  (64, 128, 3, 8.8, 0.115, 0.612, 1.06))


def pair_lib() -> ctypes.CDLL:
    return _load(_build.PAIR_GEMM)


def _pair_cost(M: int, N: int, K: int, tile: int, shares: int, groups: int = 1, tiles_of=PAIR_TILES) -> float:
    """Microseconds of a product in half precision, by the figures above.  ``groups`` as for :func:`_split_cost`."""
    bm, bn, held, fixed, alone, loaded, late = tiles_of[tile]
    tiles = -(-M // bm) if groups == 1 else M // bm + (groups + 1) // 2
    full, rest = divmod(tiles * -(-N // bn) * shares, COMPUTE_UNITS * held)
    steps = -(-K // (32 * shares)) * 2
    cost = fixed + full * loaded * steps + ((alone + (loaded - alone) * (rest / (COMPUTE_UNITS * held)) ** late) * steps if rest else 0.0)
    return max(cost, 3.0 + N * K * 4 / 5.5e6) + (shares * M * N * 4 / 4.6e6 if shares > 1 else 0.0)


def pair_plan(M: int, N: int, K: int, gated: bool = False) -> Tuple[int, int, float]:
    """(tile, shares, estimated microseconds) of :func:`pair_gemm`."""
    return _pair_plan(_whole(M), N, K, gated)


def _pair_shares(K: int, shares: int) -> int:
    """How many of ``shares`` shares of whole stages of 32 columns are not empty."""
    return -(-K // (-(-K // (32 * shares)) * 32))


@functools.lru_cache(maxsize=4096)
def _pair_plan(M: int, N: int, K: int, gated: bool) -> Tuple[int, int, float]:
    plans = [(t, s) for t in range(2 if gated else 4) for s in ((1,) if gated else (1, 2, 3, 4, 6, 8, 12)) if s == 1 or K // s >= 256]
    sums = _pair_shares(K, min((_pair_cost(M, N, K, t, s, 1, PAIR_SUM_TILES), t, s) for t, s in plans)[2])
    cost, tile, shares = min((_pair_cost(M, N, K, t, s), t, s) for t, s in plans if _pair_shares(K, s) * PAIR_SUMS[t] >= sums)
    return tile, shares, cost


def pair_holds(N: int, K: int) -> bool:
    """Whether a float32 matrix [N, K] is kept as pairs of halves beside its rows: one that :func:`pair_gemm` takes (whole
    vectors of four, bytes counted in 31 bits) and that is large enough for a product of a few thousand rows to go there."""
    return K % 4 == 0 and K >= 128 and N >= 32 and 1 << 18 <= N * K and (N + 31) * (K + 31) < 1 << 29


def _pair_planes(rows: int, K: int, device) -> Tuple[torch.Tensor, torch.Tensor]:
    return (torch.empty(rows * -(-K // 32) * 128, dtype=torch.uint8, device=device), torch.empty(rows, 2, dtype=torch.int32, device=device))


def pair_weight_bytes(N: int, K: int) -> int:
    """Bytes of what :func:`pair_weight` makes of a matrix [N, K]: as many as the matrix, and eight a row."""
    rows = -(-N // 32) * 32
    return rows * (-(-K // 32) * 128 + 8)


def pair_weight(rows: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """The float32 matrix [N, K] as :func:`pair_gemm` reads it: its numbers as two halves each, scaled by a power of two a
    row, and for every row int32 (that power, how many of its numbers are small beside its largest)."""
    N, K = rows.shape
    _gpu(rows, "w", torch.float32)
    if K % 4 or rows.data_ptr() % 16 or (N + 31) * (K + 31) >= 1 << 29:
        raise KernelError(f"pairs of halves are not made of a matrix [{N}, {K}] at this address")
    planes, info = _pair_planes(-(-N // 32) * 32, K, rows.device)
    _check(pair_lib().ni_pair_weight(_ptr(rows), _ptr(planes), _ptr(info), N, K, _stream()), "pair_weight")
    return planes, info


def pair_rows(x: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """The same of the rows of x [M, K], in another order and with the count of the numbers that are not small."""
    M, K = x.shape
    _gpu(x, "x", torch.float32)
    if K % 4 or x.data_ptr() % 16 or M * (K + 31) >= 1 << 29:
        raise KernelError(f"pairs of halves are not made of rows [{M}, {K}] at this address")
    planes, info = _pair_planes(M, K, x.device)
    _check(pair_lib().ni_pair_rows(_ptr(x), _ptr(planes), _ptr(info), M, K, _stream()), "pair_rows")
    return planes, info


class HalvedRows:
    """Float32 rows ``x`` [M, K] that a norm also left as pairs of halves (``planes`` and ``info``, what :func:`pair_rows` makes of
    them), for the products behind it.  A part that ``takes_halved`` is given one; whatever does not go to :func:`pair_gemm`
    reads ``x``."""

    __slots__ = ("x", "planes", "info")

    def __init__(self, x: torch.Tensor, planes: torch.Tensor, info: torch.Tensor):
        self.x, self.planes, self.info = x, planes, info

    @property
    def shape(self):
        return self.x.shape

    @property
    def dtype(self):
        return self.x.dtype

    @property
    def device(self):
        return self.x.device


def rows_of(x):
    """The rows themselves of what may be :class:`HalvedRows`."""
    return x.x if isinstance(x, HalvedRows) else x


def _halves_of(x):
    """(rows, planes, info) of rows or :class:`HalvedRows`."""
    return (x.x, x.planes, x.info) if isinstance(x, HalvedRows) else (x, *pair_rows(x))


def add_rmsnorm_halved(h: torch.Tensor, pending: Optional[torch.Tensor], weight: torch.Tensor, eps: float) -> HalvedRows:
    """``h += pending`` and ``rmsnorm(h) * weight`` in float32, as rows and as pairs of halves.  ``pending`` [T, d] or [S, T, d]."""
    T, d = h.shape
    _gpu(h, "h", torch.float32)
    _gpu(weight, "weight", torch.float32, (d,))
    out = torch.empty(T, d, dtype=torch.float32, device=h.device)
    addends = 1
    if pending is not None:
        addends = pending.shape[0] if pending.dim() == 3 else 1
        _gpu(pending, "pending", torch.float32, (addends, T, d) if pending.dim() == 3 else (T, d))
    if (d % 32 or d > 8192 or T * (d + 31) >= 1 << 29
            or (h.data_ptr() | weight.data_ptr() | (0 if pending is None else pending.data_ptr())) % 16):
        add_rmsnorm(h, pending, weight, eps, out)
        return HalvedRows(out, *pair_rows(out))
    planes, info = _pair_planes(T, d, h.device)
    _check(core().ni_add_rmsnorm_halves(_ptr(h), _ptr(pending), addends, ctypes.c_size_t(T * d), _ptr(weight), _ptr(out), _ptr(planes), _ptr(info),
                                        T, d, ctypes.c_float(eps), _stream()), "add_rmsnorm_halves")
    return HalvedRows(out, planes, info)


def merge_pair_rows_ok(T: int, H: int, hd: int, part_o: torch.Tensor, out: torch.Tensor) -> bool:
    """Whether :func:`merge_pair_rows` takes rows of ``H`` heads of ``hd``: they wait in registers, eight numbers a thread and chunk."""
    return (out.dtype == torch.float32 and T > 0 and hd % 8 == 0 and H * hd <= 8192 and T * (H * hd + 31) < 1 << 29
            and (part_o.data_ptr() | out.data_ptr()) % 16 == 0)


def merge_pair_rows(part_o: torch.Tensor, part_ml: torch.Tensor, out: torch.Tensor, H: int, hd: int, runs: int) -> HalvedRows:
    """The key runs of an attention, ``part_o`` float32 [T, H, runs, hd] with (maximum, sum) in ``part_ml`` [T, H, runs, 2], merged into ``out``
    [T, H * hd] and left as pairs of halves as well."""
    T = out.shape[0]
    _gpu(out, "out", torch.float32, (T, H * hd))
    _gpu(part_o, "part_o", torch.float32)
    _gpu(part_ml, "part_ml", torch.float32)
    if part_o.numel() != T * H * runs * hd or part_ml.numel() != T * H * runs * 2 or not merge_pair_rows_ok(T, H, hd, part_o, out):
        raise KernelError(f"{runs} runs of {H} heads of {hd} are not merged into pairs of halves")
    planes, info = _pair_planes(T, H * hd, out.device)
    _check(pair_lib().ni_merge_pair_rows(_ptr(part_o), _ptr(part_ml), _ptr(out), _ptr(planes), _ptr(info), T, H, hd, runs, _stream()), "merge_pair_rows")
    return HalvedRows(out, planes, info)


# Operations from which a float32 product goes to pair_gemm.  Measured in recorded launches, each with another W and all its kernels
# counted (us, library : this): [2048, 2048] at 256 / 400 / 800 rows (2.1 / 3.4 / 6.7 GFLOP) 22.8 : 26.0, 38.9 : 32.0, 65.7 : 42.9;
# [3072, 2048] at 130 / 164 / 200 (1.6 / 2.1 / 2.5) 22.6 : 26.6, 30.6 : 27.5, 31.3 : 29.5; [4096, 1024] at 256 / 400 (2.1 / 3.4) 24.1 : 26.6,
# 37.0 : 31.3; [3072, 3072] at 130 / 164 (2.5 / 3.1) 30.3 : 31.3, 42.0 : 32.2; [2048, 8192] at 65 / 130 (2.2 / 4.4) 42.6 : 40.0, 63.8 : 47.6.
PAIR_FLOPS = 2.4e9
# The same where x comes as pairs of halves (:class:`HalvedRows`): the pass over x is 4 to 5 us of those figures, a norm that does its
# work takes 2 more.  [3072, 2048] at 164 rows (2.1 GFLOP) 29.8 in the library, 22.3 here and 5.0 for its shares; at 130 (1.6) both would take 22.
PAIR_FLOPS_HALVED = 2.0e9
# Steps of fewer rows than this are a portion beside running requests, launched one by one by a host that takes as long as their
# kernels: a launch and two allocations more (10 to 15 us of it) cost what the kernels gain.  Rows of more than 8,192 numbers the
# pass over x reads twice: [2048, 16384] at 69 rows (4.6 GFLOP) 44.7 in three parts, 45.5 here and 10.0 for the pass.  Steps of 68 / 96 /
# 118 tokens, all products in three parts or from the library : by the lines above alone : by these (us): the 1B shape 2,828 : 2,745 : 2,652,
# 3,114 : 2,970 : 2,876, 3,080 : 2,968 : 2,838; the 3B shape 6,845 : 6,349 : 6,279, 7,551 : 7,065 : 6,931, 7,422 : 6,923 : 6,778; 69 / 84 / 97 / 119 of
# a hybrid with routed experts 2,406 : 2,587 : 2,475, 2,496 : 2,595 : 2,471, 2,576 : 2,599 : 2,468, 2,644 : 2,594 : 2,517;
# recorded prompts of 66 / 100 / 127 tokens, the 1B shape, 2,520 : 2,336 : 2,318, 2,725 : 2,613 : 2,522, 2,808 : 2,717 : 2,531.
PAIR_FEW_ROWS = 128
PAIR_FLOPS_FEW = 4.3e9
PAIR_FLOPS_FEW_LONG = 7.5e9


def pair_wins(x, weight) -> bool:
    """Whether a float32 product of more rows than the skinny product takes goes to :func:`pair_gemm`: a matrix that is kept as
    pairs of halves and work enough to pay for the start and for the pass that makes pairs of x (:class:`HalvedRows` need none)."""
    lines = getattr(weight, "pair_lines", None)
    if lines is None:
        return False
    halved = type(x) is HalvedRows
    rows = x.x if halved else x
    return (lines[halved] <= rows.shape[0] <= lines[2] and rows.dtype == torch.float32 and rows.is_contiguous()
            and rows.data_ptr() % 16 == 0)


def takes_halved(M: int, K: int, dtype: torch.dtype, weight) -> bool:
    """Whether the product of M rows as :class:`HalvedRows` goes there."""
    lines = getattr(weight, "pair_lines", None)
    return lines is not None and lines[1] <= M <= lines[2] and dtype == torch.float32


def pair_lines(N: int, K: int) -> Tuple[int, int, int]:
    """For a matrix [N, K] that is kept as pairs of halves: the rows of x, as they are and as :class:`HalvedRows`, from which a product
    goes to :func:`pair_gemm`, and the most that it takes."""
    def rows(flops):
        return max(SKINNY_MAX_ROWS + 1, math.ceil(flops / (2 * N * K)))

    few = rows(PAIR_FLOPS_FEW if K <= 8192 else PAIR_FLOPS_FEW_LONG)
    return (few if few < PAIR_FEW_ROWS else max(PAIR_FEW_ROWS, rows(PAIR_FLOPS)), rows(PAIR_FLOPS_HALVED), ((1 << 29) - 1) // (K + 31))


def pair_gemm(x, weight, out: Optional[torch.Tensor] = None, gated: Optional[str] = None, squared: bool = False,
              plan: Optional[Tuple[int, int]] = None, addends: bool = False) -> torch.Tensor:
    """``x . weight^T`` for float32 ``x`` [M, K] (or :class:`HalvedRows`) and a :class:`Weight` [N, K] that is kept as pairs of
    halves, by three products in half precision.  The other arguments as for :func:`split_gemm`."""
    M, K = x.shape
    rows, pairs = weight.rows, weight.pairs
    if pairs is None:
        raise KernelError("this product takes a matrix that is kept as pairs of halves")
    N = rows.shape[0]
    _gpu(rows_of(x), "x", torch.float32, (M, rows.shape[1]))
    if gated is not None and (N % 64 or squared):
        raise KernelError("a gated product takes a stacked matrix of halves of whole tiles of 32 and no other activation")
    _addends_alone(addends, out, gated, squared)
    cols = N if gated is None else N // 2
    tile, shares = plan or pair_plan(M, N, K, gated is not None)[:2]
    per = -(-K // (32 * shares)) * 32
    shares = -(-K // per)                                   # no share is empty
    x, planes, info = _halves_of(x)
    if shares > 1:
        parts = torch.empty(shares, M, N, dtype=torch.float32, device=x.device)
    elif out is None:
        out = torch.empty(M, cols, dtype=torch.float32, device=x.device)
    if out is not None:
        _gpu(out, "out", torch.float32, (M, cols))
    _check(pair_lib().ni_pair_gemm(_ptr(planes), _ptr(info), _ptr(pairs[0]), _ptr(pairs[1]), _ptr(x), _ptr(rows), _ptr(parts if shares > 1 else out),
                                   M, N, K, tile, shares, per, int(gated is not None), GATED_ACTIVATIONS[gated or "silu"],
                                   int(squared and shares == 1), _stream()), "pair_gemm")
    if shares > 1:
        return parts if addends else _add_shares(parts, torch.float32, out, squared)
    return out


# ---------------------------------------------------------------- bfloat16 on the re-tiled matrix

# Tiles of the bfloat16 product: rows of x, rows of W, workgroups a compute unit holds, and in microseconds: before the
# first and behind the last 64 columns of K, for 64 columns with one workgroup on a unit, what another on the same unit adds,
# and how much of that comes at once when the first unit gets one more.  Fitted to sweeps of all tiles and shares at 65 to
# 512 rows (with SwiGLU 1,024) over the layer sizes of the 1B, 3B and 8B shapes, recorded, every launch with another W, which
# then comes from memory as it does in a step, o and down with the norm behind them: of 117 plans taken 116 are within 5 %
# of the best and the last within 9.  (Fitted to one product launched over and over, its W at hand, as these figures were
# before, the plans were 10 % above the best on average and up to 46.)
TILED_TILES = ((128, 256, 1, 4.9, 1.02, 1.10, 0.45), (128, 128, 2, 5.3, 0.56, 0.50, 0.80), (64, 128, 4, 4.7, 0.48, 0.32, 0.85),
               (64, 64, 5, 2.8, 0.385, 0.265, 0.25))


def _tiled_cost(M: int, N: int, K: int, tile: int, shares: int, addends: bool) -> float:
    bm, bn, held, fixed, one, more, jump = TILED_TILES[tile]
    groups = -(-M // bm) * -(-N // bn) * shares
    full, rest = divmod(groups, COMPUTE_UNITS * held)

    def column(n: float) -> float:                     # 64 columns with n workgroups a unit
        return one if n <= 1 else one + more * (n + jump * (math.ceil(n) - n) - 1)

    cost = fixed + -(-(K // 64) // shares) * (full * column(held) + (column(rest / COMPUTE_UNITS) if rest else 0.0))
    cost = max(cost, 3.0 + N * K * 2 / 5.5e6)
    if shares > 1:      # the shares are written and read again, by the norm behind them or by a kernel that adds them
        cost += shares * M * N * 4 / 3.3e6 + (0.1 if addends else 3.3)
    return cost


def tiled_plan(M: int, N: int, K: int, gated: bool = False, addends: bool = False) -> Tuple[int, int]:
    """(tile, shares) of :func:`tiled_gemm`."""
    return _tiled_plan(_whole(M), N, K, gated, addends)


@functools.lru_cache(maxsize=4096)
def _tiled_plan(M: int, N: int, K: int, gated: bool, addends: bool) -> Tuple[int, int]:
    return min((_tiled_cost(M, N, K, t, s, addends), t, s) for t in range(3 if gated else 4)
               for s in ((1,) if gated else (1, 2, 3, 4, 6, 8)) if s == 1 or K // s >= 256)[1:]


TILED_ROWS = 512            # rows up to which products on the re-tiled matrix are made here
TILED_ROWS_GATED = 1024     # the same with SwiGLU in the epilogue and few columns


def tiled_wins(x: torch.Tensor, weight, gated: bool = False, addends: bool = False) -> bool:
    """Whether a bfloat16 product goes to :func:`tiled_gemm`, from 65 rows (the skinny product's end) to 512.  Measured as
    ``TILED_TILES`` (us, library : this).  Its tiles are smaller than the library's: it is ahead where it is cut along K or its
    tiles are at most one a compute unit, and behind where there are so many that the library's fill the chip as well.

    Shares left to the norm (o and down of the three shapes): always.  [2048, 2048] at 65 / 256 / 512 rows 15.5 : 10.8,
    16.1 : 14.3, 18.1 : 18.7; [2048, 8192] 25.2 : 18.2, 31.6 : 24.3, 39.1 : 33.5; [4096, 14336] 52.9 : 34.0, 67.1 : 52.6, 95.8 : 79.7.

    SwiGLU in the epilogue: while the tiles are one a unit, of a large matrix to 128 rows.  [16384, 2048] at 65 / 256 / 512 rows
    23.1 : 24.0, 34.0 : 25.8, 43.9 : 41.1, [28672, 4096] at 128 rows 61.7 : 59.6 and at 192 72.7 : 82.6.  More of them are up to a
    third slower ([28672, 4096] at 512 rows 107 : 141, [16384, 3072] at 384 49.1 : 55.1).  To 1,024 rows where the smaller tiles do
    ([4096, 2048] at 600 / 1,024 rows 26.3 : 21.6, 29.1 : 22.7; the large ones: [8192, 2048] at 767 35.4 : 40.7, [16384, 2048]
    at 640 / 1,000 47.9 : 56.3, 70 : 75).

    Plain: cut into three shares and more ([4096, 14336] at 173 / 512 rows 62.1 : 48.4, 92.8 : 78.0, [3072, 8192] at 118 / 356
    27.7 : 22.2, 42.5 : 36.6), and to 256 rows while the tiles are one a unit ([6144, 4096] at 65 / 256 rows 23.1 : 19.0, 41.1 : 31.2;
    at 263 / 512 28.8 : 36.2, 36.8 : 42.5).

    Small matrices to 512 rows in every case, though the library may be up to 4 us ahead ([3072, 2048] at 131 / 343 / 512
    rows 12.3 : 13.4, 14.6 : 15.7, 15.4 : 18.7, [5120, 3072] at 512 28.8 : 32.7, gated [16384, 2048] at 341 37.8 : 39.6): a launch here
    costs the host 10 us, the library's 18, and 79 with a number of rows that it has not seen before, and a step of single
    tokens beside a portion, launched kernel by kernel, waits for the host."""
    tiles = getattr(weight, "tiles", None)
    if x.dtype != torch.bfloat16 or tiles is None:
        return False
    M, K = x.shape
    N = weight.rows.shape[0]
    if not (64 < M <= TILED_ROWS_GATED and 0 < K and K % 64 == 0 and 0 < N and N % (32 if gated else 4) == 0 and (N + 15) * K < 1 << 30
            and M * K < 1 << 30 and x.is_contiguous() and x.data_ptr() % 16 == 0):
        return False
    tile, shares = tiled_plan(M, N, K, gated, addends)
    if M <= TILED_ROWS and (addends or shares >= 3 or N * K <= (1 << 25 if gated else 1 << 24)):
        return True
    most = 256 if not gated else 128 if N * K > 1 << 26 else TILED_ROWS if tile == 0 else TILED_ROWS_GATED
    return M <= most and -(-M // TILED_TILES[tile][0]) * -(-N // TILED_TILES[tile][1]) * shares <= COMPUTE_UNITS


def tiled_gemm(x: torch.Tensor, weight, out_dtype: Optional[torch.dtype] = None, out: Optional[torch.Tensor] = None, gated: Optional[str] = None,
               squared: bool = False, addends: bool = False, plan: Optional[Tuple[int, int]] = None) -> torch.Tensor:
    """``x . weight^T`` for bfloat16 ``x`` [M, K] and a re-tiled :class:`Weight` [N, K], in bfloat16 or (``out_dtype``) float32.
    ``gated``, ``squared``, ``addends`` and ``plan`` as for :func:`split_gemm`."""
    M, K = x.shape
    tiles = getattr(weight, "tiles", None)
    if tiles is None:
        raise KernelError("this product takes a re-tiled matrix")
    N = weight.rows.shape[0]
    out_dtype = out_dtype or x.dtype
    _gpu(x, "x", torch.bfloat16, (M, weight.rows.shape[1]))
    _gpu(tiles, "tiles", torch.bfloat16)
    if gated is not None and (N % 32 or squared or out_dtype != torch.bfloat16):
        raise KernelError("a gated product takes a stacked matrix of whole tiles, no other activation, and gives bfloat16")
    _addends_alone(addends, out, gated, squared)
    if K % 64 or N % 4 or x.data_ptr() % 16 or M * K >= 1 << 30 or (N + 15) * K >= 1 << 30 or tiles.numel() != (N + 15) // 16 * 16 * K:
        raise KernelError(f"tiled_gemm does not take [{M}, {K}] x [{N}, {K}]")
    cols = N if gated is None else N // 2
    tile, shares = plan or tiled_plan(M, N, K, gated is not None, addends)
    per = -(-(K // 64) // shares)
    shares = -(-(K // 64) // per)
    if out is not None:
        _gpu(out, "out", out_dtype, (M, cols))
        if out.data_ptr() % 16:
            raise KernelError("out is not aligned to 16 bytes")
    if shares > 1:
        parts = torch.empty(shares, M, N, dtype=torch.float32, device=x.device)
    elif out is None:
        out = torch.empty(M, cols, dtype=out_dtype, device=x.device)
    _check(tile_lib().ni_tiled_gemm(_ptr(x), _ptr(tiles), _ptr(parts if shares > 1 else out), M, N, K, tile, shares, per, int(gated is not None),
                                    int(shares > 1 or out_dtype == torch.float32), GATED_ACTIVATIONS[gated or "silu"],
                                    int(squared and shares == 1), _stream()), "tiled_gemm")
    if shares > 1:
        return parts if addends else _add_shares(parts, out_dtype, out, squared)
    return out


# ---------------------------------------------------------------- bfloat16, many rows, both operands as stored

# Tiles of the product of csrc/wide_gemm.hip: rows of x, rows of W, workgroups a compute unit holds, and in microseconds: what a launch takes
# beside its steps, 64 columns of K with one workgroup alone on its unit and with all units full, and how late between the two the
# time rises (the power of the share of the units that is taken).  Fitted to sweeps of all tiles at 192 to 4,096 rows over the layer
# sizes of the 1B, 3B and 8B shapes and smaller matrices, recorded, every launch with another W: of the plans taken the average is
# 1 % above the best, the worst 30 (tiles that just outnumber the units).
WIDE_TILES = ((256, 256, 1, 8.7, 1.055, 1.509, 2.5), (128, 256, 1, 5.1, 0.633, 0.858, 3.4), (256, 128, 1, 5.0, 0.618, 0.853, 3.0),
              (128, 128, 1, 4.0, 0.320, 0.521, 1.4), (128, 128, 2, 3.8, 0.368, 0.942, 1.2))


def wide_lib() -> ctypes.CDLL:
    return _load(_build.WIDE_GEMM)


def _wide_cost(M: int, N: int, K: int, tile: int) -> float:
    """Microseconds of a product with this tile, by the figures above."""
    bm, bn, held, fixed, alone, loaded, late = WIDE_TILES[tile]
    full, rest = divmod(-(-M // bm) * -(-N // bn), COMPUTE_UNITS * held)
    return fixed + K // 64 * (full * loaded + (alone + (loaded - alone) * (rest / (COMPUTE_UNITS * held)) ** late if rest else 0.0))


def wide_plan(M: int, N: int, K: int, gated: bool = False) -> Tuple[int, float]:
    """(tile, estimated microseconds) of :func:`wide_gemm`.  The tile of which a unit holds two is for the product whose epilogue makes
    gate and up one output: where a plain product would take it the library's is ahead ([3072, 2048] at 1,300 and 1,600 rows
    26.6 : 23.5 us, 27.2 : 23.7)."""
    return _wide_plan(_whole(M), N, K, gated)


@functools.lru_cache(maxsize=4096)
def _wide_plan(M: int, N: int, K: int, gated: bool) -> Tuple[int, float]:
    cost, tile = min((_wide_cost(M, N, K, t), t) for t in range(len(WIDE_TILES) if gated else 4))
    return tile, cost


WIDE_ROWS_GATED = 257       # rows from which a product with SwiGLU goes there, and a plain one, and to how many a plain one does
WIDE_ROWS = 513
WIDE_ROWS_LAST = 2048
WIDE_FLOPS = 2e9            # operations of the smallest plain product that was measured ([2048, 1024] at 600 rows: 10.8 us in the library, 9.5 here)


# How much longer than the library's product a plain one on each tile may be estimated to take, by where its results go: few tiles are estimated too
# high, the larger ones less so, the largest too low.  Of 289 products (17 matrices, 520 to 2,048 rows) those taken with 15 % for all but the largest
# were up to 13 % behind: [5120, 3072] at 1,024 rows 40.5 : 42.3 us, to float32 39.5 : 44.7, [8192, 4096] at 700 49.4 : 53.7, at 2,048 92.0 : 96.4 on the largest,
# whose float32 results are ahead of the library's ([8192, 2048] at 2,048 64.2 : 58.0).  With these [2048, 8192] at
# 1,400 is, by 4 %, and to float32 [6144, 4096] and [6144, 2048] at 1,024, by 6 to 7 (52.3 : 55.8, 30.8 : 32.6); a narrower line would leave [3072, 2048] at 2,045
# to the library, 34.2 : 35.3 (this : library) inside a prompt.  Where an epilogue goes on with the sums (onto the stream, squared) a kernel behind the
# product is saved, and a rounding before it.
WIDE_SLACK = {"bfloat16": (0.9, 1.08, 1.08, 1.15), "float32": (1.0, 1.05, 1.05, 1.15), "epilogue": (1.0, 1.15, 1.15, 1.15)}


def wide_wins(x: torch.Tensor, rows: torch.Tensor, gated: bool = False, to: str = "bfloat16") -> bool:
    """Whether the bfloat16 product ``x . rows^T`` goes to :func:`wide_gemm`: where it is estimated to take no longer than the library's
    product (with the SwiGLU kernel behind it): 5 to 8 us, 1 us for 1.33 GFLOP, and where its tiles are few 1.5 us for 1,024 elements of K (plain
    products of no more tiles than units by ``WIDE_SLACK``; past 8,192 elements of K, where the library is faster than that, 3 % at most).  ``to``: where
    the results go, a key of that table.  Measured in recorded launches, each with another W (us, library : this; cards differ by 10 %):

    SwiGLU in the epilogue, from 257 rows: [16384, 2048] at 400 / 512 / 900 / 1,024 / 1,300 / 1,600 / 1,999 / 3,000 / 4,096 rows 41 : 34,
    44 : 36, 64 : 58, 68 : 58, 99 : 90, 113 : 102, 121 : 111, 183 : 157, 239 : 211 (the tiled product 37 at 400 and 39 at 512 rows),
    [16384, 3072] at 512 / 1,024 / 1,999 62 : 52, 95 : 79, 172 : 152, [28672, 4096] at 512 / 1,999 108 : 102, 391 : 373, [4096, 2048] at
    600 / 1,024 / 1,999 25 : 17, 29 : 21, 42 : 31.  Not where the tiles just outnumber the units ([16384, 2048] at 600 rows 49 : 56,
    [16384, 3072] 67 : 74), and to 512 rows only on its larger tiles (a small matrix, [4096, 2048] at 512 rows, takes 19 in the smallest, 16 by
    the tiled product; [16384, 3072] at 350 is 5 % behind, 48 : 51, but the library's way rounds gate and up before it multiplies them); to 256 rows the tiled product is as fast or faster (26 : 28).

    Plain, from 513 rows (the tiled product's end) to 2,048: [2048, 8192] at 1,024 / 1,600 / 2,045 50 : 58, 66 : 58, 70 : 63, [2048, 2048] at
    800 / 1,300 / 1,600 / 2,045 15.4 : 14.8, 20.6 : 15.9, 20.7 : 17.1, 21.6 : 18.4, [3072, 2048] at 1,024 / 1,300 / 2,045 20.6 : 16.3,
    24.1 : 24.3, 28.4 : 26.4, [4096, 4096] at 1,024 / 2,045 40.7 : 35.5, 59.1 : 56.1; the results in float32, [2048, 2048] at 2,045 23.4 : 20.6,
    [3072, 2048] 28.7 : 29.0, [4096, 2048] 37.6 : 33.5, [8192, 2048] 64.2 : 57.5.  More tiles than units end in a round that few of them fill, where the
    library takes other tiles ([6144, 2048] at 2,045 48 : 55, [8192, 2048] at 1,600 49 : 56), and rows of 14,336 elements are slower here
    ([4096, 14336] at 900 / 1,300 / 1,400 116 : 122, 154 : 170, 152 : 174, but at 1,700 194 : 177); with more rows its larger ones win ([3072, 2048] at
    3,000 37 : 45, [2048, 8192] at 2,500 83 : 87)."""
    return (x.dtype == torch.bfloat16 and x.dim() == 2 and x.is_contiguous() and x.data_ptr() % 16 == 0 and wide_takes(*x.shape, rows, gated, to))


def wide_takes(M: int, K: int, rows: torch.Tensor, gated: bool = False, to: str = "bfloat16") -> bool:
    """The same of M aligned rows of K elements."""
    if rows.dtype != torch.bfloat16 or rows.dim() != 2:
        return False
    N = rows.shape[0]
    if not ((WIDE_ROWS_GATED <= M if gated else WIDE_ROWS <= M <= WIDE_ROWS_LAST) and 0 < K and K % 64 == 0 and 0 < N and N % (32 if gated else 16) == 0
            and N * K < 1 << 30 and M * K < 1 << 30 and rows.is_contiguous() and rows.data_ptr() % 16 == 0):
        return False
    tile, cost = wide_plan(M, N, K, gated)
    library = M * N * K / 0.665e9
    if gated:
        return (M >= WIDE_ROWS or tile < 3) and cost <= 12.0 + library + 3.0 * M * N / 4.6e6
    bm, bn = WIDE_TILES[tile][:2]
    slack = WIDE_SLACK[to][tile]
    if -(-M // bm) * -(-N // bn) > COMPUTE_UNITS:
        slack = min(slack, 1.0)
    if K > 8192 and to != "epilogue":
        slack = min(slack, 1.03)
    return 2.0 * M * N * K >= WIDE_FLOPS and cost <= slack * (5.0 + library + 1.5e-3 * K)


WIDE_FEW_COLUMNS = 32000
WIDE_FEW_ROUND = 65536       # columns that the chip holds tiles of at once: two tiles of 128 a unit, or one of 256


def wide_few_wins(M: int, K: int, rows: torch.Tensor) -> bool:
    """Whether 17 to 64 plain bfloat16 rows go to :func:`wide_gemm` on a matrix as stored, as the head over the vocabulary is, with float32 results: where
    the tiles fill their rounds, as far as the library does no better.  Measured with matrices that the caches do not hold (us, library : this, 17 / 32 / 64 rows):
    rows of 2,048: 32,000 columns 30.9 : 31.1, 31.0 : 31.2, 32.4 : 32.2; 36,864 39.9 : 43.4, 40.7 : 45.1, 41.9 : 47.1; 49,152 49.3 : 47.9, 50.0 : 48.5, 53.9 : 51.2;
    128,256 118.5 : 112.2, 120.9 : 115.8, 130.6 : 124.1.  4,096: 32,000 61.3 : 63.0, 61.8 : 63.6, 63.8 : 64.3; 66,560 122.5 : 134.1, 125.1 : 135.8, 131.1 : 144.6; 128,256
    202.5 : 203.8, 208.4 : 209.6, 223.9 : 223.1; 131,072 234.8 : 191.7, 241.8 : 195.5, 254.3 : 204.3.  3,072: 32,000 38.9 : 52.2, 39.3 : 54.1, 40.6 : 58.4; 65,536
    76.2 : 75.4, 79.0 : 79.0, 83.5 : 84.4; 66,560 131.0 : 105.6, 130.6 : 109.6, 92.1 : 120.3; 100,352 191.9 : 118.6, 192.4 : 123.1, 153.5 : 133.5; 128,256 161.3 : 144.7,
    167.7 : 150.7, 184.9 : 160.7.  3,584: 151,936 249.6 : 213.5, 261.9 : 217.9, 224.7 : 232.9."""
    N = rows.shape[0]
    if not (16 < M <= 64 and N >= WIDE_FEW_COLUMNS and 2048 <= K <= 4096 and K % 64 == 0 and N % 16 == 0 and N * K < 1 << 30
            and rows.dtype == torch.bfloat16 and rows.dim() == 2 and rows.is_contiguous() and rows.data_ptr() % 16 == 0):
        return False
    if K == 2048:
        return N <= 32768 or N >= 49152
    rounds, last = divmod(N - 1, WIDE_FEW_ROUND)       # full rounds, and the last column of the round behind them
    if K == 4096:
        return N >= 49152 and (rounds != 1 or last >= 24576)
    if last >= 49151:
        return True
    # a round that is not full: up to 32 rows the library is far behind
    return rounds >= 1 and (M <= 32 or last >= 32767) if K <= 3072 else rounds >= 2 and M <= 32 and last < 32767


def wide_few_tile(K: int) -> int:
    """Its tile: two workgroups a unit (64 x 128) on rows of 2,048 or 4,096 elements, one of twice the columns on those between (us, 64 x 128 : 64 x 256 on 128,256
    columns at 32 rows: 2,048 115.8 : 119.5, 2,560 133.7 : 128.9, 3,072 154.0 : 150.7, 3,584 174.4 : 170.7, 4,096 209.6 : 226.9)."""
    return 5 if K in (2048, 4096) else 6


def wide_stream_ok(M: int, K: int, dtype: torch.dtype, weight) -> bool:
    """Whether the product of M rows of K elements onto the residual stream goes to :func:`wide_stream`: by the line of a plain product with more slack,
    as a norm kernel behind it is not launched, or reads one operand less.  Measured (us, the library's product and a norm : this, its norm left half
    done : this and a norm): [2048, 2048] at 1,024 / 1,600 / 2,048 rows 21.4 : 19.0 : 21.3, 28.7 : 21.4 : 25.5, 31.7 : 23.7 : 28.4, [2048, 8192] at 1,600 / 2,048 74.4 : 62.0 :
    65.6, 81.3 : 66.9 : 71.5, [3072, 3072] at 1,024 / 2,048 37.3 : 32.0 : 36.2, 55.3 : 47.5 : 53.8, [4096, 4096] at 800 / 2,048 47.8 : 38.1 : 43.0, 78.0 : 64.5 : 74.1.  The line
    leaves out some that are ahead ([2048, 2048] at 800 20.2 : 18.9, [2048, 8192] at 1,300 62.8 : 59.4, [3072, 3072] at 800 / 1,300 35.6 : 31.2, 49.3 : 45.1, [4096, 4096] at
    600 42.4 : 36.2) with those that are not ([2048, 8192] at 600 / 1,024 46.4 : 60.6, 55.8 : 61.0, [3072, 8192] at 1,300 84.9 : 92.8)."""
    rows = getattr(weight, "rows", None)
    return rows is not None and M >= WIDE_ROWS and dtype == torch.bfloat16 and rows.shape[0] % 64 == 0 and wide_takes(M, K, rows, to="epilogue")


def wide_leaves_ok(M: int, K: int, dtype: torch.dtype, weight) -> bool:
    """Whether that product can leave the next norm's input half done: rows of 256 to 4,096 elements, whose sums of squares come in whole
    vectors of parts of 64 columns."""
    return wide_stream_ok(M, K, dtype, weight) and weight.rows.shape[0] % 256 == 0 and weight.rows.shape[0] <= 4096


def wide_stream(x: torch.Tensor, rows: torch.Tensor, h: torch.Tensor, weight: Optional[torch.Tensor] = None, tile: Optional[int] = None):
    """``h += x . rows^T`` for bfloat16 ``x`` and ``rows`` and the float32 stream ``h``.  With the ``weight`` [N] of the norm behind it
    (``h * weight`` in bfloat16, the sums of ``h^2`` over 64 columns at a time [M, N / 64]) are returned."""
    M, K = x.shape
    N = rows.shape[0]
    _gpu(x, "x", torch.bfloat16)
    _gpu(rows, "w", torch.bfloat16, (N, K))
    _gpu(h, "h", torch.float32, (M, N))
    if K % 64 or K == 0 or N % 64 or N == 0 or M == 0 or (x.data_ptr() | rows.data_ptr() | h.data_ptr()) % 16 or M * K >= 1 << 30 or N * K >= 1 << 30:
        raise KernelError(f"wide_stream does not take [{M}, {K}] x [{N}, {K}]")
    following = ss = None
    if weight is not None:
        _gpu(weight, "norm weight", torch.float32, (N,))
        if weight.data_ptr() % 16:
            raise KernelError("the norm's weight is not aligned to 16 bytes")
        following = torch.empty(M, N, dtype=torch.bfloat16, device=x.device)
        ss = torch.empty(M, N // 64, dtype=torch.float32, device=x.device)
    _check(wide_lib().ni_wide_stream(_ptr(x), _ptr(rows), _ptr(h), _ptr(weight), _ptr(following), _ptr(ss), M, N, K,
                                     wide_plan(M, N, K)[0] if tile is None else tile, _stream()), "wide_stream")
    return following, ss


def _row_norm(x, M: int, K: int):
    """(rows, sums of squares, parts, eps) of what a product of many rows is given: rows, or a :class:`ScaledInput`."""
    if isinstance(x, torch.Tensor):
        return x, None, 0, ctypes.c_float(0.0)
    _gpu(x.ss, "sums of squares", torch.float32)
    if x.ss.dim() != 2 or x.ss.shape[0] != M or not 0 < x.ss.shape[1] <= 64 or x.ss.shape[1] % 4 or x.ss.data_ptr() % 16:
        raise KernelError(f"sums of squares {tuple(x.ss.shape)} of {M} rows")
    return x.x, x.ss, int(x.ss.shape[1]), ctypes.c_float(x.norm.eps)


def wide_gemm(x, rows: torch.Tensor, out_dtype: Optional[torch.dtype] = None, out: Optional[torch.Tensor] = None, gated: Optional[str] = None,
              squared: bool = False, tile: Optional[int] = None) -> torch.Tensor:
    """``x . rows^T`` for bfloat16 ``x`` [M, K] and ``rows`` [N, K] as stored, in bfloat16 or (``out_dtype``) float32.  ``gated`` and ``squared`` as for
    :func:`split_gemm`.  ``tile``: another than :func:`wide_plan`'s.  With ``gated`` ``x`` may be a :class:`ScaledInput`."""
    M, K = x.shape
    N = rows.shape[0]
    out_dtype = out_dtype or x.dtype
    x, ss, parts, eps = _row_norm(x, M, K)
    if ss is not None and gated is None:
        raise KernelError("the plain product does not take a scaled input")
    _gpu(x, "x", torch.bfloat16)
    _gpu(rows, "w", torch.bfloat16, (N, K))
    if gated is not None and (N % 32 or squared or out_dtype != torch.bfloat16):
        raise KernelError("a gated product takes a stacked matrix of whole tiles, no other activation, and gives bfloat16")
    if K % 64 or K == 0 or N % 16 or N == 0 or M == 0 or x.data_ptr() % 16 or rows.data_ptr() % 16 or M * K >= 1 << 30 or N * K >= 1 << 30:
        raise KernelError(f"wide_gemm does not take [{M}, {K}] x [{N}, {K}]")
    cols = N if gated is None else N // 2
    if out is None:
        out = torch.empty(M, cols, dtype=out_dtype, device=x.device)
    _gpu(out, "out", out_dtype, (M, cols))
    if out.data_ptr() % 16:
        raise KernelError("out is not aligned to 16 bytes")
    if tile is None:
        tile = wide_plan(M, N, K, gated is not None)[0]
    _check(wide_lib().ni_wide_gemm(_ptr(x), _ptr(rows), _ptr(out), M, N, K, tile, int(gated is not None), int(out_dtype == torch.float32),
                                   GATED_ACTIVATIONS[gated or "silu"], int(squared), _ptr(ss), parts, eps, _stream()), "wide_gemm")
    return out


# ---------------------------------------------------------------- bfloat16, [q; k; v] with rotation and the cache's pages behind it

ROPE_PASS = 3.5, 2.2e-3      # microseconds of the kernel that rotates and stores: a launch, and a row (4.3 at 512 rows, 7.9 at 1,999, the 1B shape)
ROPE_SHARES_PASS = 3.0       # of the pass that adds a product's shares as well, beside what moving them takes


@functools.lru_cache(maxsize=4096)
def _qkv_rope_plan(M: int, N: int, K: int, hd: int, tiled: bool) -> Optional[Tuple[bool, int]]:
    """(whether on the re-tiled matrix, tile) of :func:`qkv_rope`, or None where the product and a kernel behind it are estimated to be faster."""
    ahead = ROPE_PASS[0] + ROPE_PASS[1] * M
    if M <= TILED_ROWS:
        if not tiled:
            return None
        cost, tile = min((_tiled_cost(M, N, K, t, 1, False), t) for t in range(3))
        t, shares = _tiled_plan(M, N, K, False, False)
        if shares == 1:                    # (small matrices are estimated a third too high)
            return (True, tile) if M > 256 and N * K <= 1 << 22 or cost <= _tiled_cost(M, N, K, t, 1, False) + ahead else None
        return (True, tile) if cost <= _tiled_cost(M, N, K, t, shares, True) + ROPE_SHARES_PASS else None
    if hd % 64 or 2.0 * M * N * K < WIDE_FLOPS:
        return None
    tile, cost = _wide_plan(M, N, K, False)
    return (False, tile) if cost <= 1.15 * (5.0 + M * N * K / 0.665e9 + 1.5e-3 * K) + ahead else None


def qkv_rope_plan(x, weight, hd: int, rotary_dim: int) -> Optional[Tuple[bool, int]]:
    """How the product of more than 64 bfloat16 rows with the stacked matrix [q; k; v] rotates and stores in its epilogue (:func:`qkv_rope`), None where
    it does not: heads rotated whole, of whole tiles, and a product that :func:`tiled_wins` sends to the re-tiled matrix or that the
    one on the stored matrix makes in the time of the library's, with 15 % more, and the rotating kernel's.  Not so close a line as a plain product's: that
    kernel is given rows that were rounded already, the epilogue rounds once (logits of a prompt of 300 tokens of the 1B shape against 64 bits 1.56e-2, by
    the kernel 1.80e-2).  Measured in recorded launches, each with another W (us, the library's product and the kernel : this): [3072, 2048] (the 1B shape) at 600 /
    1,024 / 1,300 / 1,999 / 2,500 / 4,096 rows 20.9 : 19.6, 28.3 : 20.9, 32.3 : 29.4, 36.9 : 30.7, 40.7 : 34.2, 58.0 : 52.5, but at 3,000 45.7 : 48.6; [5120, 3072] (3B) at 600 /
    1,024 / 1,500 / 1,999 / 2,500 36.7 : 29.9, 45.8 : 44.9, 55.7 : 46.9, 73.6 : 69.0, 82.0 : 73.5, but at 800 / 1,800 41.7 : 43.4, 63.3 : 69.2; [6144, 4096] (8B) at 600 / 1,024 / 1,200 /
    2,500 46.8 : 39.9, 59.5 : 56.0, 66.6 : 59.1, 104.6 : 101.7, but at 800 / 1,500 / 1,600 / 1,800 52.7 : 53.8, 83.5 : 88.0, 78.8 : 89.7, 88.8 : 95.0.  With float32 results of the library and the pass that
    rounds once those are 53, 79, 81, 91 and the 3B ones 45 and 66: no better way at most sizes."""
    if not isinstance(x, torch.Tensor):
        return wide_rope_plan(*x.shape, x.dtype, weight, hd, rotary_dim) if hasattr(x, "ss") else None
    if x.dtype != torch.bfloat16 or x.dim() != 2 or hd % 32 or rotary_dim != hd:
        return None
    M, K = x.shape
    rows = getattr(weight, "rows", None)
    if M <= SKINNY_MAX_ROWS or rows is None or rows.dtype != torch.bfloat16 or not (x.is_contiguous() and x.data_ptr() % 16 == 0):
        return None
    N = rows.shape[0]
    if K == 0 or K % 64 or N == 0 or N % hd or M * K >= 1 << 30 or (N + 15) * K >= 1 << 30:
        return None
    if M <= TILED_ROWS:
        if not tiled_wins(x, weight):
            return None
    else:
        return wide_rope_plan(M, K, x.dtype, weight, hd, rotary_dim)
    return _qkv_rope_plan(_whole(M), N, K, hd, getattr(weight, "tiles", None) is not None)


def qkv_whole(x, weight) -> bool:
    """Whether the product of 65 to 512 bfloat16 rows with the stacked matrix [q; k; v], where it does not rotate itself, is made whole, with float32
    results for the pass that rounds once (:func:`rope_kv_write_shares` of one share), instead of cut into shares for it: where :func:`tiled_wins`
    would leave it to the library if nothing behind it added shares.  Cutting pays where that is done in any case or the tiles fill no chip;
    [6144, 4096] at 320 / 400 / 448 / 512 rows (us, shares : this) 37.1 : 35.6, 44.3 : 39.7, 45.5 : 40.8, 46.8 : 42.6 (rounded rows and the rotating kernel 34.4, 35.7, 37.3,
    41.0), but cut without that, at 352 / 384, 37.9 : 41.9, 38.9 : 42.0, as [5120, 3072] at 256 / 384 22.7 : 36.4, 26.3 : 28.8."""
    return x.dtype == torch.bfloat16 and tiled_wins(x, weight, addends=True) and not tiled_wins(x, weight)


def wide_rope_plan(M: int, K: int, dtype: torch.dtype, weight, hd: int, rotary_dim: int) -> Optional[Tuple[bool, int]]:
    """:func:`qkv_rope_plan` of M aligned rows past those of the tiled product, also where they are a :class:`ScaledInput`."""
    rows = getattr(weight, "rows", None)
    if rows is None or dtype != torch.bfloat16 or rows.dtype != torch.bfloat16 or M <= TILED_ROWS or hd % 64 or rotary_dim != hd:
        return None
    N = rows.shape[0]
    if (K == 0 or K % 64 or N == 0 or N % hd or M * K >= 1 << 30 or (N + 15) * K >= 1 << 30 or not rows.is_contiguous() or rows.data_ptr() % 16):
        return None
    return _qkv_rope_plan(_whole(M), N, K, hd, False)


def qkv_rope(x, weight, positions: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, slot_mapping: Optional[torch.Tensor],
             kpool: Optional[torch.Tensor], vpool: Optional[torch.Tensor], H: int, KVH: int, hd: int, plan: Tuple[bool, int]) -> torch.Tensor:
    """``x . weight^T`` for many bfloat16 rows and the stacked matrix [q; k; v]: returns the rotated queries [M, H * hd]; rotated keys and
    plain values go into the pools ([pages, KVH, page_size, hd]) at ``slot_mapping`` (below zero, or absent: not stored).  ``plan`` as
    :func:`qkv_rope_plan` gives it.  On the stored matrix ``x`` may be a :class:`ScaledInput`."""
    M, K = x.shape
    given = x
    on_tiles, tile = plan
    rows, tiles = weight.rows, weight.tiles
    x, ss, parts, eps = _row_norm(x, M, K)
    if ss is not None and on_tiles:
        raise KernelError("the product with the re-tiled matrix does not take a scaled input")
    _gpu(x, "x", torch.bfloat16)
    _gpu(rows, "w_qkv", torch.bfloat16, ((H + 2 * KVH) * hd, K))
    _gpu(positions, "positions", torch.int32, (M,))
    _gpu(cos, "cos", torch.float32)
    _gpu(sin, "sin", torch.float32, cos.shape)
    N = rows.shape[0]
    matrix = tiles if on_tiles else rows
    if (hd % (32 if on_tiles else 64) or 2 * cos.shape[1] != hd or K == 0 or K % 64 or M * K >= 1 << 30 or (N + 15) * K >= 1 << 30 or matrix is None
            or (on_tiles and tiles.numel() != N * K) or (x.data_ptr() | matrix.data_ptr()) % 16):
        raise KernelError(f"qkv_rope does not take [{M}, {K}] x [{N}, {K}] with heads of {hd}, of which {2 * cos.shape[1]} are rotated")
    page_size = 1
    if slot_mapping is not None:
        _gpu(slot_mapping, "slot_mapping", torch.int32, (M,))
        if kpool is None or vpool is None:
            raise KernelError("a slot mapping needs both pools")
        _gpu(kpool, "kpool", torch.bfloat16)
        _gpu(vpool, "vpool", torch.bfloat16, kpool.shape)
        if not (kpool.dim() == 4 and kpool.shape[1] == KVH and kpool.shape[3] == hd):
            raise KernelError(f"pool must be [pages, {KVH}, page_size, {hd}], is {tuple(kpool.shape)}")
        page_size = kpool.shape[2]
    if _off_vectors(cos, sin):
        cos, sin = cos.clone(), sin.clone()
    if slot_mapping is not None and _off_vectors(kpool, vpool):
        # keys and values to pages of one token, and from there as the kernel behind a product stores them
        whole = [torch.empty(M, KVH, 1, hd, dtype=torch.bfloat16, device=given.device) for _ in range(2)]
        q = qkv_rope(given, weight, positions, cos, sin, torch.arange(M, dtype=torch.int32, device=given.device), *whole, H, KVH, hd, plan)
        rope_kv_write(torch.cat([q, *(t.view(M, -1) for t in whole)], dim=1), positions, None, None, slot_mapping, kpool, vpool, H, KVH, hd)
        return q
    q = torch.empty(M, H * hd, dtype=torch.bfloat16, device=x.device)
    launch, norm = (tile_lib().ni_tiled_qkv_rope, ()) if on_tiles else (wide_lib().ni_wide_qkv_rope, (_ptr(ss), parts, eps))
    _check(launch(_ptr(x), _ptr(matrix), _ptr(q), _ptr(positions), _ptr(cos), _ptr(sin), _ptr(slot_mapping), _ptr(kpool), _ptr(vpool), M, K, H, KVH, hd,
                  page_size, tile, *norm, _stream()), "qkv_rope")
    return q


# ---------------------------------------------------------------- routed experts

def _grouped_plan(places: int, N: int, K: int, groups: int) -> Tuple[float, int]:
    return _grouped_tiles(_whole(places), N, K, groups)


@functools.lru_cache(maxsize=1024)
def _grouped_tiles(places: int, N: int, K: int, groups: int) -> Tuple[float, int]:
    return min((_split_cost(places, N, K, t, 1, groups), t) for t in range(len(SPLIT_TILES)))


def _grouped_pair_plan(places: int, N: int, K: int, groups: int) -> Tuple[float, int]:
    return _grouped_pair_tiles(_whole(places), N, K, groups)


@functools.lru_cache(maxsize=1024)
def _grouped_pair_tiles(places: int, N: int, K: int, groups: int) -> Tuple[float, int]:
    return min((_pair_cost(places, N, K, t, 1, groups), t) for t in range(len(PAIR_TILES)))


def _experts_in_pairs(places: int, w_up, w_down, d: int, per: int, ff: int) -> bool:
    """Whether both products of routed experts are made in half precision: matrices that are kept as pairs of halves, an
    expert's rows of up whole tiles of 32 and its columns of down whole stages."""
    return (getattr(w_up, "pairs", None) is not None and getattr(w_down, "pairs", None) is not None and d % 32 == 0 and ff % 32 == 0
            and per % 32 == 0 and places * max(d, ff) < 1 << 29)


def experts_grouped_wins(x, w_up, w_down, top: int, experts: int) -> bool:
    """Whether routed experts of float32 rows go expert by expert (:func:`experts_grouped`) instead of as two dense
    products over all experts: by the estimates of :func:`split_plan` or :func:`pair_plan`, with 25 us for the lists and the sums
    beside the passes over the entries' rows.  1,500 rows of 2,048 elements, four of sixteen experts of 1,024: 290 us for the two
    products against 960 (in three parts)."""
    up, down = getattr(w_up, "rows", w_up), getattr(w_down, "rows", w_down)
    x = rows_of(x)
    M, d = x.shape
    per, ff = up.shape[0] // experts, down.shape[1] // experts
    if not (x.dtype == torch.float32 and d % 4 == 0 and ff % 4 == 0 and M * top < 1 << 24 and split_wins(x, up)
            and down.is_contiguous() and down.data_ptr() % 16 == 0):
        return False
    places = M * top
    plan, whole = (_grouped_pair_plan, pair_plan) if _experts_in_pairs(places, w_up, w_down, d, per, ff) else (_grouped_plan, split_plan)
    grouped = plan(places, per, d, experts)[0] + plan(places, d, ff, experts)[0] + 25.0 + (12.0 * d + 4.0 * per) * places / 4e6
    # (some five launches more, which a host that is behind pays for: see PAIR_FEW_ROWS)
    return grouped + (40.0 if M < PAIR_FEW_ROWS else 0.0) < whole(M, experts * per, d)[2] + whole(M, d, experts * ff)[2]


def experts_grouped(x, w_up, w_down, chosen: torch.Tensor, mix: torch.Tensor, experts: int,
                    act, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The weighted sum of every row's chosen experts, float32 [T, d]: the entries (token, expert) are put in the order of
    their experts, each expert multiplies its own tokens' rows, and a token's results are added in the order in which it
    chose.  ``w_up`` [E * per, d], ``w_down`` [d, E * ff], tensors or :class:`Weight`; ``act(up [entries, per], weights [entries, 1])``
    gives the hidden rows [entries, ff].  An index of E or more in ``chosen`` int32 [T, top] names an expert that is not among these."""
    up_rows, down_rows = getattr(w_up, "rows", w_up), getattr(w_down, "rows", w_down)
    halved, x = x, rows_of(x)
    T, d = x.shape
    top, E = chosen.shape[1], experts
    places = T * top
    if up_rows.shape[0] % E or down_rows.shape[1] % E:
        raise KernelError("the matrices are not whole experts")
    per, ff = up_rows.shape[0] // E, down_rows.shape[1] // E
    _gpu(x, "x", torch.float32)
    _gpu(up_rows, "w_up", torch.float32, (E * per, d))
    _gpu(down_rows, "w_down", torch.float32, (d, E * ff))
    _gpu(chosen, "chosen", torch.int32, (T, top))
    _gpu(mix, "mix", torch.float32, (T, top))
    if d % 4 or ff % 4 or any(t.data_ptr() % 16 for t in (x, up_rows, down_rows)):
        raise KernelError("rows of the experts' products are not aligned to 16 bytes")
    pairs = _experts_in_pairs(places, w_up, w_down, d, per, ff)
    ints = torch.empty(E + 1 + 2 * places, dtype=torch.int32, device=x.device)
    offsets, rows, place = ints[:E + 1], ints[E + 1:E + 1 + places], ints[E + 1 + places:]
    weights = torch.empty(places, 1, dtype=torch.float32, device=x.device)
    lib = tile_lib()
    _check(lib.ni_expert_lists(_ptr(chosen), _ptr(mix), T, top, E, _ptr(offsets), _ptr(rows), _ptr(weights), _ptr(place), _stream()), "expert_lists")
    up = torch.empty(places, per, dtype=torch.float32, device=x.device)
    if pairs:
        _pair_grouped(halved, w_up, up, offsets, rows, E, False)
    else:
        _check(lib.ni_split_gemm_grouped(_ptr(x), _ptr(up_rows), _ptr(up), places, per, d, _ptr(offsets), _ptr(rows), E, ctypes.c_size_t(per * d), d,
                                         _grouped_plan(places, per, d, E)[1], _stream()), "experts_up")
    hidden = act(up, weights)
    _gpu(hidden, "hidden", torch.float32, (places, ff))
    y = torch.empty(places, d, dtype=torch.float32, device=x.device)
    if pairs:
        _pair_grouped(hidden, w_down, y, offsets, None, E, True)
    else:
        _check(lib.ni_split_gemm_grouped(_ptr(hidden), _ptr(down_rows), _ptr(y), places, d, ff, _ptr(offsets), None, E, ctypes.c_size_t(ff), E * ff,
                                         _grouped_plan(places, d, ff, E)[1], _stream()), "experts_down")
    if out is None:
        out = torch.empty(T, d, dtype=torch.float32, device=x.device)
    _gpu(out, "out", torch.float32, (T, d))
    _check(lib.ni_gather_entries(_ptr(y), _ptr(place), _ptr(out), T, d, top, _stream()), "gather_entries")
    return out


def _pair_grouped(x, weight, out: torch.Tensor, offsets: torch.Tensor, rows: Optional[torch.Tensor], experts: int, down: bool) -> None:
    """``out[p] = x[rows[p]] . W_e^T`` for the places p of every expert's list; its rows of W behind the others' or (``down``) beside them."""
    places, N = out.shape
    K = x.shape[1]
    x, planes, info = _halves_of(x)
    _check(pair_lib().ni_pair_gemm_grouped(_ptr(planes), _ptr(info), _ptr(weight.pairs[0]), _ptr(weight.pairs[1]), _ptr(x), _ptr(weight.rows), _ptr(out),
                                           places, N, K, _ptr(offsets), _ptr(rows), experts, int(down),
                                           _grouped_pair_plan(places, N, K, experts)[1], _stream()), "pair_gemm_grouped")
