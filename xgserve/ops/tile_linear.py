"""Products of many rows (prompt steps) on csrc/mixers/tile_linear.h: the sizes they run at, and where the library's stay.

`tile_plan` prices every tile and split of K of the kernel with a model that was fitted to 13 900 timings on an MI355X (2 590 products
of 52 weights of 512 to 18944 in K and 32 to 37888 in N, 65 to 6000 rows, cold weights), of the kernel whose load ring ended with each
tile of the result. Over these its choice was 0.6 % slower than the fastest form that was timed in the mean and 19 % at most. Of the kernel
as it is, whose ring runs through the tiles, 144 products of 16 weights were timed (65 to 6000 rows, all forms within half of the cheapest
price): 0.8 % in the mean, 9 % at most (251 x 4096 x 14336 48.7 us, 44.9 on 256 x 128 in eight parts). The figures that follow are of the
fit. A step of 64 of K costs a workgroup its products or, of few rows, its reads:
weights come from memory, rows from L2, at the rate at which its outstanding loads return (ops.seqmix._rows_cols has the same for a few
rows). Without that the smallest tiles looked cheaper than they are: us, 224 x 4096 x 4096 27.1 -> 21.9, 768 x 2048 x 8192 50 -> 37,
288 x 18560 x 4096 75 -> 60; of 483 products, whose plan this changed, the times are 8 % less in the mean, 11 % more at most. A
product's time steps up with every round of tiles that is begun, so there are many sizes: (5, 8), (8, 6), (7, 6), (6, 6), (7, 4) and
(5, 4) beside the ten that were there take 2 % off the mean of 144 products of 80 to 5000 rows, and, us, cold weights: 2521 x 4096 x
14336 243 -> 213 (256 tiles of 160 x 256, where 192 x 256 left 32 of 256 workgroups out), 2521 x 2048 x 8192 79 -> 74, 3100 x 6144 x
4096 139 -> 126, 1024 x 18560 x 4096 148 -> 130, 700 x 6144 x 4096 43 -> 38.
"""
from __future__ import annotations

import array
import functools
from typing import Optional

import torch
import torch.autograd.forward_ad as _fwd_ad
from torch._C._functorch import is_functorch_wrapped_tensor as _is_transformed
from torch.overrides import _get_current_function_mode_stack as _function_modes
from torch.utils._device import DeviceContext

from ._native import is_f32, mixers, native_device, on_current_device, stream_ptr
from .linear import PendingSum, cu_count

# rows and columns of a workgroup's tile / 32 -> us per 64 of K where its products bound it, and per tile
_TILES = {(8, 8): (1.184, 5.47), (7, 8): (1.130, 3.75), (6, 8): (0.967, 4.90), (5, 8): (0.868, 3.15), (4, 8): (0.883, 1.35),
          (8, 6): (1.055, 3.27), (7, 6): (0.911, 3.74), (6, 6): (0.790, 3.47), (8, 4): (0.793, 2.94), (7, 4): (0.707, 2.70),
          (6, 4): (0.648, 2.68), (5, 4): (0.556, 2.47), (4, 4): (0.499, 2.39), (3, 4): (0.410, 3.21), (4, 2): (0.309, 2.69),
          (3, 2): (0.319, 0.02)}
# ... and where its reads do: us per 64 of K for 32 rows, for 32 columns (of weights that one row of tiles reads: with n of them n^-1/4 of
# it), and for the smallest tile besides
_X_READ, _W_READ, _SMALL = 0.0371, 0.1037, 0.0913
_SUM, _PART = 4.91, 0.230                    # us of the launch that adds the parts, and for each of them
_PART_BYTES, _OUT_BYTES = 2.51e6, 2.52e6   # bytes per us: fp32 parts (there and back), the result
_SPLITS = (1, 2, 3, 4, 6, 8, 12, 16)
_SPLIT_K, _SPLIT_TILES = 256, 540           # a part's least K; parts of all tiles at most (a bound on the slabs: 2.1 tiles per CU)

PAIR_NONE, PAIR_HALVES, PAIR_BLOCKS = 0, 1, 2   # rows of a gated weight: [gate | up], or 16 gate rows, 16 up rows, ...
COLUMNS_END = 1 << 22                       # 128 rows of fp32 results stay below 2^31 bytes
TILE_ROWS_MIN = 65                          # (up to 64 rows the weights are streamed past them: rows_linear)


def _table(kind: str, *rows):
    """(address, entries) of numbers that stay for the process, for the native search."""
    a = array.array(kind, [v for r in rows for v in r])
    _KEPT.append(a)
    return a.buffer_info()


_KEPT: list = []
_PRICES = _table("d", (_X_READ, _W_READ, _SMALL, _SUM, _PART, _PART_BYTES, _OUT_BYTES, _SPLIT_K, _SPLIT_TILES))[0]
_TILE_ROWS = _table("d", *(t + p for t, p in _TILES.items()))[0]
_SPLIT_ROWS = _table("i", _SPLITS)[0]


@functools.lru_cache(maxsize=8192)   # (csrc/mixers/tile_plan.cpp: 2 us for a new size, 60 in Python)
def tile_plan(M: int, N: int, K: int, cus: int = 256):
    """(rows / 32, columns / 32, parts of K) of an [M, K] . [N, K]^T product."""
    return mixers().tile_plan(_TILE_ROWS, len(_TILES), _SPLIT_ROWS, len(_SPLITS), _PRICES, M, N, K, cus)


# Tiles of the experts' products; offsets of all experts are looked through for a tile's, so there is a bound on their number
# (their prices are a fit of their own: rows are gathered, and most experts end in a part of a tile; with them the weights' reads are a
# constant, so the time of the tiles alone decides)
_GROUPED = {(8, 8): (1.098, 0.02), (7, 8): (0.995, 0.63), (6, 8): (0.868, 0.86), (4, 8): (0.694, 1.11), (6, 4): (0.527, 1.55),
            (4, 4): (0.401, 1.88), (3, 4): (0.331, 1.95)}
GROUPED_EXPERTS_MAX = 64
_SHARES = (-1.2, -0.9, -0.6, -0.2, 0.2, 0.6, 0.9, 1.4)   # eight quantiles of an expert's rows, in units of their spread ...
_SPREAD = 0.55                                            # ... from the mean, in units of the mean
_GROUPED_ROWS = _table("d", *(t + p for t, p in _GROUPED.items()))[0]
_QUANTILES = _table("d", [z * _SPREAD for z in _SHARES])[0]


@functools.lru_cache(maxsize=4096)
def grouped_plan(pairs: int, E: int, N: int, K: int, cus: int = 256):
    """(rows / 32, columns / 32) for `pairs` rows shared out among E experts' [N, K] weights: `tile_plan`'s prices, the tiles counted at
    eight quantiles of an expert's rows. Routers share out unevenly (0.5 to 0.6 of the mean from it, over experts); with the square root
    of the mean instead, tiles that just hold the mean were taken, and the larger experts' second ones made a round of their own. Cold
    weights, both products, router and shared expert, us: 8 experts of 2 x 2048 x 2048, 300 tokens 131 -> 124; of 2 x 3584 x 4096 256 ->
    241, 400 tokens 290 -> 276 (either product's change alone)."""
    return mixers().grouped_plan(_GROUPED_ROWS, len(_GROUPED), _QUANTILES, len(_SHARES), pairs, E, N, K, cus)


def library_better(M: int, N: int, K: int) -> bool:
    """Whether the library's plain product (nothing behind it) is the faster one (us, library against this kernel): long ones, which run
    at the card's power limit, where the library's needs less of it, by 1 to 10 % (28672x4096, 8192 rows 1284 against 1370; 4096x4096,
    4001 rows 95 against 98; 16384x2048, 2048 rows 103 against 115; 6144x4096, 8192 rows 279 against 305; but 4096x4096, 3072 rows 81
    against 76), as long as no columns are left over beside its tiles of 256
    (10304x2048, 4001 rows 182 against 146; 18560x4096, 2048 rows 347 against 272) and these fill their rounds of the chip to three
    quarters (below, at 0.6, 6144x4096, 3100 rows 166 against 126; 4096x14336, 2521 rows 249 against 237;
    4096x4096, 5000 rows 140 against 129; up to 1792 rows 4096x14336, 1536 rows 188 against 150; 6144x4096, 700 rows 52 against 40). Its narrow
    products of few rows are up to 1 us faster on the card (2048x2048, 65 rows 9.4 against 9.7, 256 rows 10.7 against 11.5), and some of
    middle size by as much (6144x4096, 512 rows 38.8 against 40.2), others no longer (4096x4096, 256 rows 23.3 against 22.7; 18560x4096, 400
    rows 71 against 68), but not in steps. Eager ones of few rows wait for the host, of which the library's call takes 31 us and this kernel's
    10: with the faster of both for every product, 96 rows, Vizonex "1b" 868 -> 1159 us, Dofivik 1300 -> 1507; from 400 rows on within
    1 %. Replayed ones of 96 and 160 rows are up to 2 % slower with it, of 256 rows up to 2 % faster."""
    tiles = -(-M // 256) * (N // 256)
    return N % 256 == 0 and M > 1792 and 4 * tiles >= 3 * 256 * -(-tiles // 256)


def forward_only(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor]) -> bool:
    """Whether nothing follows these tensors through the call or stands before it: no graph, no tangents, no function transform, no
    tracing, function or dispatch mode (a default device alone is none: it makes tensors), no autocast, which chooses the product's
    type, no tensor type of its own. (A product on a kernel of this library has no derivative and no operator to record; torch's has.)"""
    if _fwd_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack() > 0 or torch.jit.is_tracing() \
            or torch.compiler.is_compiling() or torch.is_autocast_enabled(x.device.type):
        return False
    if torch._C._len_torch_function_stack() > 0 and any(type(m) is not DeviceContext for m in _function_modes()):
        return False
    for t in (x, w, bias):
        if t is not None and (type(t) not in (torch.Tensor, torch.nn.Parameter) or _is_transformed(t)):
            return False
    return not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad or (bias is not None and bias.requires_grad)))


def tile_plan_of(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, pairs: int = PAIR_NONE,
                 plain: bool = False):
    """The plan of x . w^T on the tile kernel, or None: bfloat16 on the current device, more than 64 rows of whole 16-byte pieces, K in
    whole steps of 64, whole groups of columns, nothing that wants a derivative; `plain` products only where the library's is not
    faster. What is refused here goes to torch, which refuses what it cannot do."""
    if not (native_device(x) and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.dim() == 2
            and w.device == x.device and w.dim() == 2 and x.shape[0] >= TILE_ROWS_MIN and forward_only(x, w, bias)
            and on_current_device(x)):
        return None
    (M, ldk), (N, K) = x.shape, w.shape
    if ldk != K or K < 64 or K % 64 or N < 8 or N % (32 if pairs == PAIR_BLOCKS else 8) or not w.is_contiguous() or \
            x.stride(1) != 1 or x.stride(0) < K or x.stride(0) % 8 or (x.data_ptr() | w.data_ptr()) % 16:
        return None
    # (a lane's offsets are 32 bits: of the whole weight, of a tile's rows and of its results; tiles are counted in an int)
    if 2 * N * K >= 1 << 32 or 512 * x.stride(0) >= 1 << 32 or N >= COLUMNS_END or M * N >= 1 << 40:
        return None
    if bias is not None and not (pairs == PAIR_NONE and bias.device == x.device and bias.dtype in (torch.float32, torch.bfloat16)
                                 and bias.shape == (N,) and bias.is_contiguous() and bias.data_ptr() % 16 == 0):
        return None
    return None if plain and library_better(M, N, K) else tile_plan(M, N, K, cu_count(x.device))


def tile_linear(plan, x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, act: int = 0, p0: float = 0.0,
                p1: float = 0.0, pairs: int = PAIR_NONE) -> torch.Tensor:
    """act(x . w^T + bias) on `plan` (`tile_plan_of`); act: ops.seqmix's ACT_..., gated ones with `pairs`."""
    M, (N, K), (fm, fn, S) = x.shape[0], w.shape, plan
    out = torch.empty(M, N // 2 if pairs else N, dtype=x.dtype, device=x.device)
    part = torch.empty(S * M * N, dtype=torch.float32, device=x.device) if S > 1 else None
    mixers().tile_linear(x.data_ptr(), x.stride(0), w.data_ptr(), 0 if bias is None else bias.data_ptr(),
                         bias is not None and is_f32(bias), 0 if part is None else part.data_ptr(), out.data_ptr(), M, N, K, S, act,
                         pairs, float(p0), float(p1), fm, fn, cu_count(x.device), stream_ptr())
    return out


def tile_parts(plan, x: torch.Tensor, w: torch.Tensor) -> PendingSum:
    """x . w^T on a `plan` with K in parts, which the next kernel adds."""
    M, (N, K), (fm, fn, S) = x.shape[0], w.shape, plan
    part = torch.empty(S, M, N, dtype=torch.float32, device=x.device)
    mixers().tile_linear(x.data_ptr(), x.stride(0), w.data_ptr(), 0, False, part.data_ptr(), 0, M, N, K, S, 0, PAIR_NONE, 0.0, 0.0,
                         fm, fn, cu_count(x.device), stream_ptr())
    return PendingSum(part, S)
