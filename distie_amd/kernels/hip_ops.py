"""`HipOps`: the kernel surface on hand-written HIP kernels for gfx950.

The kernels live in shared libraries built from `distie_amd/csrc` and are called (`calls.py`)
with raw device pointers on torch's current HIP stream, so they take part in
stream order and in graph capture like any other launch. torch is the allocator and the
stream/graph owner; the only library routine on this path is the matrix product for
large bfloat16 operands (the reference leaves its products to a library too).

Constructing `HipOps` without a GPU, without hipcc-built libraries, or for a head size
the kernels refuse, raises: there is no fallback.
"""

from __future__ import annotations

import ctypes
import functools
import logging
from typing import Dict, Optional

import numpy as np
import torch

from ..csrc import build
from . import calls
from .interface import BatchMeta, Ops, RouteRule

_log = logging.getLogger(__name__)

_F32, _BF16 = 0, 1
_CODES = {torch.float32: _F32, torch.bfloat16: _BF16}
_P = ctypes.c_void_p
_I = ctypes.c_int
_L = ctypes.c_int64
_F = ctypes.c_float


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


class KernelError(RuntimeError):
    pass


def _code(t: torch.Tensor) -> int:
    try:
        return _CODES[t.dtype]
    except KeyError:
        raise KernelError(f"kernels take float32 and bfloat16 tensors, not {t.dtype}") from None


def _check(status: int, name: str) -> None:
    if status == 0:
        return
    if status < 0:
        raise KernelError(f"{name}: the kernel refuses these sizes or types")
    raise KernelError(f"{name}: launch failed with HIP error {status}")


def _written(t: torch.Tensor):
    """How often `t` has been written in place, as far as anyone can know: torch's own count (every in-place
    torch operation on the tensor or on a view of it) and the count of this module's kernels that write their
    argument (`_mark_written`)."""
    return (t._version, getattr(t, "_distie_version", 0))


def _mark_written(t: torch.Tensor) -> None:
    t._distie_version = getattr(t, "_distie_version", 0) + 1


class _NotATensorYet:
    """What `HipOps` hands out in place of a tensor. Anything asked of it that only a tensor has raises
    with the way out, instead of an AttributeError far from the cause."""

    def __getattr__(self, name):
        raise KernelError(f"{type(self).__name__} is a result of the HIP kernels that is not a tensor yet (asked for "
                          f".{name}): a part that computes on the values itself calls ops.dense(value) first")


class PartialSums(_NotATensorYet):
    """The result of a matrix product whose reduction was cut into slices: float32
    [slices, rows, columns], to be added in order by whoever reads it. `linear` returns it for
    small batches (a sum across workgroups inside the product would cost more than the product);
    `add_rmsnorm`, `silu_mul` and `rope_kv_write` add the slices while they read, every other
    operation sees the finished sum through `HipOps.dense`."""

    def __init__(self, data: torch.Tensor, dtype: torch.dtype) -> None:
        self.data = data
        self.dtype = dtype                  # the dtype the finished sum would have
        self.shape = data.shape[1:]
        self.device = data.device

    @property
    def slices(self) -> int:
        return self.data.shape[0]


class PendingNorm(_NotATensorYet):
    """rmsnorm(residual) * weight, not computed yet: for steps of few rows the product that reads it computes
    it itself, in front of its own work (`distie_decode_norm_product`); anything else sees the finished
    tensor through `HipOps.dense`. Valid as long as the residual it was made from is unchanged: a write in
    place by torch (also through a view) or by one of this module's kernels between `rmsnorm` and the use is
    found out and raises, instead of a norm of the wrong values."""

    def __init__(self, residual: torch.Tensor, weight: torch.Tensor, eps: float, dtype: torch.dtype) -> None:
        self.residual = residual
        self.weight = weight
        self.eps = float(eps)
        self.dtype = dtype
        self.shape = residual.shape
        self.device = residual.device
        self.version = _written(residual)

    def check(self) -> None:
        if _written(self.residual) != self.version:
            raise KernelError("a normed value was used after the residual stream it was made from had changed")


class PendingProduct(_NotATensorYet):
    """x W^T + bias for few rows of x, not computed yet: if the next thing that happens to it is the sum into
    the residual stream, the product adds itself to the stream in place (`distie_decode_product_residual`) and
    never exists as a tensor; anything else sees the finished tensor through `HipOps.dense`."""

    def __init__(self, x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> None:
        self.x = x
        self.weight = weight
        self.bias = bias
        self.dtype = x.dtype
        self.shape = torch.Size((x.shape[0], weight.shape[0]))
        self.device = x.device


class NormedSum(_NotATensorYet):
    """scale * sum_i rmsnorm(terms[i]) * weights[i], not computed yet: if what happens to it next is the norm behind
    its sub-layer and the sum into the residual stream, one kernel does all of it (`distie_norm_chain`); anything else
    sees the finished float32 tensor through `HipOps.dense`."""

    def __init__(self, terms, weights, eps: float, scale: float) -> None:
        self.terms, self.weights, self.eps, self.scale = terms, weights, eps, scale
        self.dtype = torch.float32
        self.shape = terms[0].shape
        self.device = terms[0].device


class LayerTail:
    """What is left of a layer behind attention (`HipOps.layer_tail`), done in one launch (`distie_layer_chain`) once it is known whether
    another layer's q/k/v product follows."""

    def __init__(self, ops, residual, mixed, out_weight, norm_weight, eps, gate_up_weight, down_weight, scratch) -> None:
        self.ops, self.residual, self.mixed, self.scratch = ops, residual, mixed, scratch
        self.weights = (out_weight, gate_up_weight, down_weight)
        self.norm = (norm_weight, float(eps))

    def finish(self):
        return self.ops._layer_chain(self, None)[0]

    def finish_into(self, norm_weight, eps, weight, bias, meta, group, k_cache, v_cache, inv_freq, num_heads, num_kv_heads, head_dim,
                    write):
        held = getattr(weight, "_distie_rotary", None)
        if held is None or held[1] != (num_heads, num_kv_heads, head_dim) or inv_freq is None or \
                2 * inv_freq.shape[0] != head_dim or k_cache.dtype != torch.bfloat16 or self.mixed.dtype != torch.bfloat16:
            return None
        M, C = self.residual.shape
        N, ops = weight.shape[0], self.ops
        if weight.shape[1] != C or N != (num_heads + 2 * num_kv_heads) * head_dim or norm_weight.dtype not in _CODES or \
                tuple(norm_weight.shape) != (C,) or M != meta.num_tokens or meta.groups[group].slots.shape[0] != M or \
                (bias is not None and (bias.dtype != torch.float32 or bias.shape[0] != N)) or \
                held[0].numel() != ops._packed_elements(N, C, False) or not ops._chain_fits(M, C, *self._inner(), N):
            return None
        ops._own(norm_weight, bias, k_cache, v_cache, inv_freq, meta.groups[group].slots)
        ops._check_cache(k_cache, v_cache, num_kv_heads, meta.block_size, head_dim)
        return ops._layer_chain(self, (norm_weight, float(eps), held[0], bias, ops._rope_table(meta, inv_freq),
                                       meta.groups[group].slots, k_cache, v_cache, num_heads, num_kv_heads, head_dim,
                                       meta.block_size, 1 if write else 0))

    def _inner(self):
        return self.mixed.shape[1], self.weights[2].shape[1]


class HipOps(Ops):
    # Steps of up to FUSED_MAX_ROWS rows can run their products with the norm in front and the residual sum behind
    # folded in (six launches a layer instead of eight, no partial sums handed on). On the device that is no
    # gain: a kernel's time here is a chain of trips to memory, and the folded-in norm or the sum across a
    # workgroup's waves adds its trip to the product's own (measured at 8 rows, 1,536 wide: gate+up 18.7 us with
    # the norm against 13.4 + 4.2 us apart; down 13.2 against 8.3 us in 14 slices, since 96 workgroups pull
    # less than 1,344; q/k/v 9.0 against 5.5 + 4.2 us). Where the host bounds a step, two launches fewer a layer
    # count: steps that are launched kernel by kernel take this path, captured steps do not.
    FUSED_MAX_ROWS = 16
    FUSED_IN_CAPTURED_STEPS = False
    # float32 products (and products against weights kept in float32) of up to ROWS_MAX_ROWS rows stream the weights
    # through `gemv_rows` (FMAs on the vector ALU); beyond that the tiled float32 kernel
    ROWS_MAX_ROWS = 64
    # float32 products of up to 32 rows on the matrix cores (`rows_f32`), timed beside `gemv_rows` on 42 weights of 0.1 to 105
    # million elements, each from memory, with the kernel that reads the result (us, `rows_f32` / `gemv_rows`):
    #  * gated and q/k/v products, with activation, or rotation and cache write, in the epilogue: always (1 row: gate+up [128, 64]
    #    2.9 / 4.6, [9728, 896] 11.4 / 12.1, [17920, 1536] 23.7 / 26.6, q/k/v [2048, 1536] 7.7 / 11.2; 32 rows 3.8 / 6.1, 20 / 46, 45 /
    #    82, 13 / 24), but for weights below ROWS_F32_MIN_ELEMENTS, which keep the rounding of the kernel on the vector ALU;
    #  * plain ones, whose slices of K the reader has to add (`_rows_f32_take`): at up to 4 rows only long weights (1 row: [1536,
    #    1536] 8.7 / 6.9, [3584, 3584] 19.5 / 14.1, [1536, 8960] 18.7 / 17.2, [5120, 20480] 97 / 89, but [2560, 10240] 29.8 / 32.0,
    #    [4096, 16384] 54 / 60; 2 to 4 rows: [4096, 10240] 37 / 38 to 43, [2048, 8192] 20 / 19 to 22); at 5 to 8 rows, where the vector
    #    ALU takes another group of rows, weights past ROWS_F32_EIGHT_ELEMENTS ([2048, 2048] 9.7 / 9.3, [1536, 8960] 18.9 / 23.7);
    #    beyond, weights of enough rows to fill the chip ([512, 2048] 6.9 / 6.4 at 12 rows, 8.5 / 7.2 at 24; [640, 1600] 7.0 / 7.5 at
    #    12, 8.8 / 7.8 at 24, where the vector ALU takes three groups of eight rows, and 8.9 / 10.3 at 32, four; [768, 768] 7.5 / 7.5
    #    and 8.2 / 9.8; [1536, 1536] 9.4 / 11.4 and 10.7 / 14.4).
    ROWS_F32_MIN_ELEMENTS = 64 << 10
    ROWS_F32_FEW_ELEMENTS = 20 << 20
    ROWS_F32_EIGHT_ELEMENTS = 4 << 20
    # bfloat16 products by rows of x: up to SKINNY_MAX_ROWS the weights are streamed by one wave per block
    # of 16 weight rows, x straight from memory (above that, the library's tiles are faster);
    SKINNY_MAX_ROWS = 16
    # on a packed copy the one-wave kernel is the faster one only up to 8 rows: at 9 to 16 rows every wave reads all
    # 16 rows of x beside its weights, and the kernel that shares x through LDS takes over (decode step at batch 12
    # and 16: 1.5B shape 1.77 -> 1.66 and 1.95 -> 1.81 ms, 7B shape 4.34 -> 3.91 and 4.92 -> 4.14 ms; at batch 8 and
    # below the one-wave kernel is level or ahead)
    ONE_WAVE_MAX_ROWS = 8
    # with a packed copy of the weight, more rows go through the kernel that shares the x tile of a workgroup in
    # LDS, in passes over the weight: up to PACKED_MAX_ROWS in a captured step (measured in the decode step: 9 %
    # faster than the library at 72 rows, 5 % at 96, 4 % slower at 128), and up to PACKED_MAX_ROWS_EAGER in a step
    # that is launched kernel by kernel, which the host bounds at these sizes: the library's products cost it
    # 18 us each and the activation and rotation kernels beside them more launches (a portion of n tokens behind
    # 512, this way and through the library, 1.5B shape: 100: 2.8 and 3.4 ms, 160: 3.1 and 3.4, 200: 3.6 and 3.5,
    # 224: 3.7 and 3.5).
    # A weight of more than PACKED_LARGE_ELEMENTS (64 MB) is not held by the memory-side cache from one pass to the
    # next: a pass takes up to 96 rows, and every further one reads the weight from memory again, which the library
    # does once. Which is faster then goes by the weight's shape (7B shape at 128 rows, the packed kernels in two
    # passes and the library's best kernel by timing, with the same flush of the caches before each: gate+up
    # [37888, 3584] 144 and 115 us, the head [152064, 3584] 535 and 297, down [3584, 18944] 75 and 91):
    #  * K longer than the weight has rows (down): the packed kernels, whose K is cut into slices, up to
    #    PACKED_MAX_ROWS_LARGE rows, captured or not;
    #  * more rows than K (gate+up, the head, a large q/k/v): one pass, PACKED_MAX_ROWS_LARGE_WIDE rows. Once the
    #    library's kernels were timed for a class of row counts (`library_timed_rows`, set by the engine's start with
    #    `tune_products`), the library takes over from 65 rows on (PACKED_MAX_ROWS_LARGE_WIDE_TIMED): untimed, its
    #    choice is good at one row count and poor at the next. 7B shape, decode step at batch 72, 80, 96, 112, 128,
    #    160, 192: 6.4, 6.6, 7.3, 8.1, 8.4, 10.4, 10.9 ms timed; 6.6, 6.8, 8.0, 8.6, 9.6, 11.7, 12.0 untimed; and with
    #    every large weight on the packed kernels up to 192 rows 6.6, 6.8, 8.0, 9.2, 9.7, 11.9, 13.3. At 24 to 64 rows
    #    the timed library is 1-3 % ahead as well (gate+up rounded to bfloat16 before the activation): left as it is.
    # The 1.5B shape's weights are small, its head large: its captured step is the same either way.
    PACKED_MAX_ROWS = 96
    PACKED_MAX_ROWS_LARGE = 192
    PACKED_MAX_ROWS_LARGE_WIDE = 96
    PACKED_MAX_ROWS_LARGE_WIDE_TIMED = 64
    PACKED_MAX_ROWS_EAGER = 192
    PACKED_LARGE_ELEMENTS = 32 << 20
    # or, for a weight of at most this many elements (too few row blocks to occupy the chip that way),
    # through the one-wave kernel once per 16 rows of x
    ROW_GROUPS_MAX_ELEMENTS = 4 << 20
    # the q/k/v product with rotation and cache write in its epilogue exists per 16 rows only; from so many rows on a
    # weight above that size runs on the wide kernel instead, with rotation and cache write as the kernel behind it
    # (7B shape, decode step: 1.5 % slower at 24 rows, the same at 32 and 48, 2.7 % faster at 64)
    WIDE_QKV_MIN_ROWS = 49
    # ... and that kernel takes more than 32 rows in two passes of 32 over a weight of at most this many elements
    # (64 MB: the second pass reads it from the memory-side cache; much larger ones would come from memory twice)
    TWO_PASS_MAX_ELEMENTS = 32 << 20
    # ... and a larger one is read once per pass: as few passes as the kernel's 96 rows a pass allow, of equal size
    # (7B shape: decode step at batch 80 6.8 ms in one pass of 80 rows, 7.7 as 64 + 16; at batch 96 8.1 and 8.3;
    # a portion of 160 tokens 7.4 ms in two passes of 80 and 8.4 in three of 64, 64 and 32)
    WIDE_PASS_MAX_BLOCKS = 6
    # From TILES_MIN_ROWS rows of x on, products on a packed copy whose K is a multiple of 64 run in tiles
    # (`packed_tiles.hip`) where that is faster than the passes above and than the library, or level with them
    # (`_tiles_take`). Measured on 46 weights of 0.6 to 141 million elements, 33 to 2,048 rows, every weight from memory, the
    # kernel that reads the result included (us, tiles / what there was: passes up to 96 rows, beyond them the library's
    # first choice and its best by timing):
    #  * whole K: while every workgroup has a compute unit to itself and the tile is one of the two small ones. Past that the
    #    library's tiles are level or ahead: [512, 1536] x [1536, 1536] 12 / 13, 13; [1200, 1536] 17 / 19, 19; [1400, 1536] 21
    #    / 21, 20; [900, 8192] x [3072, 8192] on 96 x 128 68 / 64, 66. 96 x 128 pays where the weight has more rows than K
    #    and the library was not timed: [576, 1024] x [4352, 1024] 12.7 / 15.0, 12.4;
    #  * K cut, for readers that add the slices (TILES_CUT_ROWS): K at least twice as long as the weight has rows up to
    #    TILES_LONG_ROWS: [97, 8960] x [1536, 8960] 15 / 26, 26; [320, 8960] 24 / 33, 34; [1024, 8960] 47 / 53, 55; other
    #    weights up to TILES_CUT_MAX_ROWS: [256, 3584] x [3584, 3584] 21 / 24, 22; [384, 1536] x [1536, 1536] 13 / 12, 12. Up to 64
    #    rows the passes are level or ahead but for weights of few rows: [64, 8960] x [1536, 8960] 15 / 16; [64, 18944] x
    #    [3584, 18944] 41 / 36; [64, 5120] x [5120, 5120] 25 / 22. From 65 to 80 rows a pass over a weight of more than 64 MB holds them
    #    all: [80, 18944] x [3584, 18944] 42 / 41, in one round of small tiles [80, 11008] x [4096, 11008] 30 / 42. Small
    #    weights (TILES_SMALL_ELEMENTS) only against the library's first choice: [97, 1024] x [1024, 1024] 8 / 11, 8;
    #  * K cut beyond TILES_LONG_ROWS, for the large weights of a portion of a prompt (TILES_PORTION_ELEMENTS) as far as they were
    #    measured, against the library's first choice: [2048, 18944] x [3584, 18944] 296 / 382, 268; [1600, 27648] x
    #    [5120, 27648] 571 / 681, 416; not [1800, 27648] 560 / 455, 470 nor [1400, 11008] x [4096, 11008] 160 / 149, 148. An engine
    #    that timed the library's kernels for a portion of these rows stays with them. (`large_tiles` has taken over what begins at
    #    multiples of 16 bytes; this is for the rest;)
    #  * gated products, which save the activation's kernel: [64, 1536] x [17920, 1536] 20 / 22; [192, 1536] 28 / 30, 29; [301,
    #    1536] 34 / 34, 35; [193, 2048] x [16384, 2048] 32 / 31, 32: up to TILES_MAX_GATED_WORK, and where the host bounds the step,
    #    or one pass of 96 rows is what there is, as far as they are level, TILES_LEVEL_GATED_WORK. Weights of up to
    #    TILES_SMALL_GATED elements from 81 rows on where one round of tiles holds them ([88, 1024] x [8192, 1024] 9 / 10;
    #    [88, 896] x [9728, 896] 12 / 11), or beyond the passes' rows; up to TILES_MAX_SMALL_GATED_WORK ([512, 1024] x [8192,
    #    1024] 21 / 22, 23; [832, 1024] 28 / 26, 27);
    #  * q/k/v with rotation and cache write in the epilogue: one round of 64 x 64 tiles: [80, 3584] x [4608, 3584] 20 / 22;
    #    [512, 1536] x [2048, 1536] 11 / 14, 13; in tiles of 64 x 128 the epilogue costs what it saves ([640, 1536] 18 / 17, 17)
    #    but for large weights beside an untimed library ([224, 3584] x [4608, 3584] 30 / 37, 27). Weights of up to
    #    ROW_GROUPS_MAX_ELEMENTS have kernels of 16 rows, up to 96 rows of a captured step and 192 of another ([96, 1024] x [1536,
    #    1024] 9.1 / 6.7): from there on.
    TILES_MIN_ROWS = 33
    TILES_MIN_ROTARY_ROWS = 80
    TILES_MAX_WORK = 4.5e9
    TILES_MAX_GATED_WORK = 6.45e9
    TILES_LEVEL_GATED_WORK = 8.5e9
    TILES_MAX_SMALL_GATED_WORK = 4.8e9
    TILES_SMALL_GATED = 10 << 20
    TILES_SMALL_ELEMENTS = 2 << 20
    TILES_CUT_ROWS = 65
    TILES_FEW_WEIGHT_ROWS = 2048
    TILES_CUT_MAX_ROWS = 320
    TILES_LONG_ROWS = 1024
    TILES_PORTION_ELEMENTS = 56 << 20
    TILES_PORTION_ROWS = 2048
    TILES_PORTION_WORK = 2.3e11
    TILES_LARGE_ROTARY = 12 << 20
    # In a step that is launched kernel by kernel a product of the library's costs the host 10 us more than one of these, the
    # kernel behind it for activation or rotation its own launch, and the passes' rules take longer to walk through. Where
    # weights are small (TILES_SMALL_GATED) the host bounds such a step up to about TILES_HOST_ROWS, whatever its kernels take:
    # tiles then go up to TILES_MAX_WORK (a layer of the Mepapel decoder of width 1024, 899 rows: gate+up in tiles 29 us instead
    # of 28, the step 20 us a layer shorter; a prompt of 100 tokens, 1.5B shape, q/k/v in tiles 10 us instead of 9, the step
    # 2,245 us instead of 2,302).
    TILES_HOST_ROWS = 2048
    # (A weight that no role was named for stays with the passes: who reads its product is not known.)
    # From LARGE_FEW_ROWS + 1 rows on, products on a packed copy run in the tiles of `large_tiles.hip` where those are the faster ones
    # (`_large_take`). Which is told by the rate, in TFLOP/s, that the count behind their plan comes to; measured on 25 weights of
    # 0.9 to 136 million elements and 27 row counts, in a captured graph, with the kernels that read the result (us, these tiles /
    # what there was, `packed_tiles` or the library's first choice with the kernels behind it):
    #  * gated: from LARGE_GATED_RATE on ([65, 1536] x [17920, 1536] 19 / 22, [301, 1536] 27 / 35, [2048, 1536] 111 / 128; [2048,
    #    3584] x [37888, 3584] 451 / 570, [72, 3584] 56 / 74; [160, 1024] x [8192, 1024] 12 / 13, [2048, 1024] 37 / 44), with gelu, squares
    #    or max(z, 0) on the gate as well (gelu [2048, 1024] x [8192, 1024] 39 / 46, [1802, 2048] x [16384, 2048] 122 / 124);
    #  * with rotation and cache write in the epilogue: beyond one round of the 64 x 64 tiles of `packed_tiles` ([512, 1536] x
    #    [2048, 1536] 17 / 12, [576, 1536] 17 / 18, [1152, 1536] 19 / 25, [2048, 1536] 24 / 26; [416, 2048] x [3072, 2048] 20 / 20, [512,
    #    2048] x [2560, 2048] 23 / 21), with K beyond LARGE_ROTARY_SHORT_K one of their 64 x 128 tiles ([352, 3072] x [4096, 3072] 32 / 25,
    #    [512, 3072] 33 / 29, [576, 3072] 31 / 33; [512, 2560] x [3328, 2560] 30 / 27, [640, 2560] 30 / 31), for large weights
    #    LARGE_ROTARY_ROWS ([480, 3584] x [4608, 3584] 37 / 36, [800, 3584] 38 / 45, [1280, 3584] 50 / 54), up to LARGE_ROTARY_WORK
    #    products: alone [1802, 3584] takes 66 / 70 and [2048, 3584] 78 / 71, but in a serving step of 2,025 tokens of the 7B shape the
    #    kernel here takes 78 us a layer and the library's with the one behind it 68 + 17: they suffer more from the clock that the
    #    products around them leave (the whole step 24.07 ms / 24.15, runs differ by as much); [1024, 4096] x [6144, 4096] 58 / 61,
    #    [2304, 4096] 136 / 106; [672, 5120] x [7168, 5120] 60 / 69, [2048, 5120] 166 / 143. Many rows of [2048,
    #    1536]: 2,304 29 / 31, 3,072 32 / 32, 4,096 40 / 40;
    #  * plain, for readers that add the slices of K: K at least twice as long as the weight has rows from LARGE_LONG_RATE on
    #    ([512, 8960] x [1536, 8960] 34 / 31, [576, 8960] 30 / 33, [2048, 8960] 66 / 83; [193, 18944] x [3584, 18944] 48 / 58, [2048,
    #    18944] 271 / 300), and past TILES_LONG_ROWS, where `packed_tiles` ends, LARGE_LONG_RATE_BEYOND ([1024, 4096] x [1024,
    #    4096] 22 / 21, [1280, 4096] 23 / 27); others from LARGE_SHORT_RATE on ([256, 3584] x [3584, 3584] 19.5 / 19, [301, 3584] 23 /
    #    26; [1408, 1536] x [1536, 1536] 24 / 23, [1536, 1536] 21 / 23), weights of 2,048 rows and up to
    #    ROW_GROUPS_MAX_ELEMENTS from LARGE_SHORT_RATE_SMALL on ([1536, 2048] x [2048, 2048] 30 / 28, [1667, 2048] 27 / 30);
    #  * rotating ones and those of readers that add slices up to LARGE_ROWS rows; up to LARGE_MAX_ROWS where K is five times as long
    #    as the weight has rows, and up to LARGE_MANY_ROWS_WORK products ([2304, 8192] x [2048, 8192] 88 / 96, [4096, 8192] 141 / 132,
    #    [8192, 8192] 246 / 216; [3072, 8960] x [1536, 8960] 93 / 109, [4096, 8960] 116 / 119, [8192, 8960] 207 / 195; [8192, 1536] x
    #    [2048, 1536] with rotation 79 / 58). Steps, us, with this line / without: 1.5B shape, 8,000 tokens 28,040 / 28,690; 7B shape,
    #    4,096 tokens 49,220 / 50,600. The gated ones win at 8,192 rows, too ([8192, 1536] x [17920, 1536] 386 / 446);
    #  * other plain ones from LARGE_PLAIN_RATE on ([1024, 2048] x [2048, 2048] 17 / 15, [1152, 2048] 17 / 20), weights of four times as
    #    many rows as K from LARGE_WIDE_RATE on ([352, 1280] x [5440, 1280] 15.5 / 14.2, [416, 1280] 14.3 / 14.8; [256, 1536] x [6528, 1536]
    #    17.5 / 13.6, [416, 1536] 16.3 / 16.7; [160, 2560] x [10880, 2560] 25 / 23, [176, 2560] 24 / 39), with K of up to LARGE_WIDE_SHORT_K
    #    from LARGE_WIDE_SHORT_RATE on ([400, 1024] x [4352, 1024] 11 / 10, [480, 1024] 11 / 12; [720, 768] x [3264, 768] 9.1 / 10.7), up to
    #    LARGE_DENSE_WORK products, from where the library is the faster one ([900, 2048] x [8448, 2048] 36 / 40, [1024, 2048] 42 / 39, [2048, 2048] 76 / 66).
    # A single row of tiles (65 to 192 rows), half of the compute units or fewer with one: such a tile takes 0.5 us and more for every
    # 64 k, however idle the rest is, and the smaller tiles and passes of before, which spread over more units, are ahead where K is
    # long: beyond LARGE_IDLE_K ([88, 2560] x [13824, 2560] 27 / 25, [160, 3072] x [16384, 3072] 39 / 35; plain [128, 3072] x [13056,
    # 3072] 33 / 29, [192, 3584] x [15232, 3584] 45 / 35; with K = 2,048 level: [88, 2048] x [16384, 2048] 24.3 / 23.6, [128, 2048]
    # 24.5 / 25.6), a quarter of them at any K ([128, 1536] x [8192, 1536] 18.0 / 13.2). Not where all that is left are passes over the
    # weight, which are much slower than tiles there ([160, 2560] x [10880, 2560] in those of packed_tiles 22, [176, 2560] in passes 39).
    LARGE_IDLE_K = 2048
    # Up to LARGE_FEW_ROWS rows the kernel takes smaller tiles, and no count stands behind their plan (28 weights, 1 to 64 rows; what
    # there was are the passes over the packed copy and `packed_tiles`):
    #  * gated: from LARGE_FEW_GATED_ROWS rows on, weights of less than LARGE_FEW_GATED_ELEMENTS from LARGE_FEW_CUT_ROWS on ([8, 1536]
    #    x [17920, 1536] 12.5 / 13.0, [9, 1536] 13.4 / 14.7, [32, 1536] 13.6 / 16.0, [64, 1536] 15.5 / 20.5; [16, 2048] x [16384, 2048]
    #    15.1 / 16.0; [64, 3584] x [37888, 3584] 53 / 66; [12, 1536] x [8192, 1536] 8.4 / 8.6, [12, 1280] x [7168, 1280] 7.6 / 7.2; [16, 1024] x
    #    [8192, 1024] 7.0 / 6.8, [17, 1024] 7.1 / 7.5; [9, 512] x [4096, 512] 4.6 / 4.4, [20, 512] 4.6 / 5.3);
    #  * plain, for readers that add slices: LARGE_FEW_CUT_ROWS rows of large weights ([16, 3584] x [3584, 3584] 12.5 / 12.3, [20,
    #    3584] 12.7 / 13.2, [64, 3584] 14.4 / 16.1; [32, 8192] x [2048, 8192] 13.0 / 15.2; [64, 11008] x [4096, 11008] 25 / 37; [24,
    #    8960] x [1536, 8960] 13.0 / 13.0; [64, 2048] x [2048, 2048] 9.6 / 9.3);
    #  * the heads of large vocabularies, LARGE_FEW_HEAD_ELEMENTS, from LARGE_FEW_CUT_ROWS rows on ([16, 1536] x [151936, 1536] 88 /
    #    89, [20, 1536] 92 / 93, [64, 1536] 99 / 116; [24, 3584] x [151936, 3584] 197 / 206; of [152064, 3584] in a decoding step 199 / 212,
    #    behind 2,025 rows of prompts 206 / 216; [32, 2048] x [32768, 2048] 26.5 / 27.5 and [64, 2048] 27.5 / 27.4).
    LARGE_FEW_ROWS = 64
    LARGE_FEW_GATED_ROWS = 9
    LARGE_FEW_GATED_ELEMENTS = 10 << 20
    LARGE_FEW_CUT_ROWS = 17
    LARGE_FEW_LONG_ELEMENTS = 16 << 20
    LARGE_FEW_SHORT_ELEMENTS = 12 << 20
    LARGE_FEW_HEAD_ELEMENTS = 128 << 20
    # Several products with inputs of their own share a launch of these tiles, as far as that was measured (four of [C, C] and a
    # narrow unrounded one, which stays with the library at 12 us, us together / one by one in the library: C = 512, 300 rows 10 /
    # 29; 1,024, 450 rows 18 / 42; 2,048, 33 rows 20 / 48, 1,802 rows 67 / 103; 3,072, 2,048 rows 147 / 185).
    LARGE_EACH_WORK = 8e10
    LARGE_MIN_ROWS = 9
    LARGE_GATED_RATE = 240.0
    LARGE_ROTARY_RATE = 150.0
    LARGE_ROTARY_ROWS = 416
    LARGE_ROTARY_SHORT_K = 2048
    LARGE_ROTARY_WORK = 4e10
    LARGE_ROWS = 2304
    LARGE_MAX_ROWS = 4096
    LARGE_MANY_ROWS_WORK = 1.3e10
    LARGE_LONG_RATE = 515.0
    LARGE_LONG_RATE_BEYOND = 380.0
    LARGE_SHORT_RATE = 316.0
    LARGE_SHORT_RATE_SMALL = 440.0
    LARGE_PLAIN_RATE = 480.0
    LARGE_WIDE_RATE = 390.0
    LARGE_WIDE_SHORT_RATE = 350.0
    LARGE_WIDE_SHORT_K = 1024
    LARGE_DENSE_WORK = 1.65e10
    # What a cut product costs beyond its slices where the reader of the result cannot add them itself (the readers of a
    # layer's output projections can)
    ADDS_SLICES = ("attn_out", "down")
    SUM_SLICES_US = 4.5
    # attention over a portion of a prompt: from so many visible keys on, the walk over the keys is cut into so
    # many parts that run side by side (measured at 12 heads of 128, 2,048 new tokens: 3 parts are best up to
    # 4,096 keys, 5 at 8,192, 8 from 16,384 on; the kernel takes up to 16)
    PREFILL_PARTS = ((1024, 3), (8192, 5), (16384, 8))
    PREFILL_WORKGROUPS = 512         # as many workgroups a short portion's attention should have, if its keys allow
    # Heads of 64 and 128 in bfloat16 up to so many times the keys from which the tiled kernel's walk is cut (4,608 keys with up to 256
    # workgroups of 32 tokens, 3,584 with more): the kernel whose waves share the columns and split the keys. Tiled with its merge /
    # that one, us, 12 heads of 128: prompts of 40 tokens 6.3 / 5.6, 301 13.5 / 7.7, 1,024 27.2 / 14.0, 2,048 38.0 / 27.1, 3,500 77 /
    # 62, 300 behind 4,000 34.5 / 27.1, 600 39 / 30; beyond, 28 heads, 600 behind 4,000 76 / 81, 1,500 147 / 156 (64 heads, 600: 129 /
    # 149; heads of 64, 28 of them, 4,500 tokens 126 / 139); 12 heads, 128 behind 16,000 55 / 83
    PREFILL_WAVES_REACH = ((256, 4.5), (None, 3.5))
    # few tokens far behind are too few workgroups for either; the tiled kernel's parts are more: 64 behind 4,000 (16 heads) 23.2 /
    # 26.0, 32 behind 3,000 (8 heads) 17.4 / 19.8, 32 behind 1,500 (12 heads) 18.4 / 13.1, 100 behind 3,000 30 / 20
    PREFILL_WAVES_FEW = (96, 2560)
    # many workgroups that all walk far (keys / tokens of a portion): the tiled kernel reads them for 128 tokens at once. 40 heads, 400 behind
    # 3,100, 520 workgroups 55 / 66; 28 heads, 364 workgroups 46 / 44; 64 heads of 64, 1,000 behind 2,000, 2,048 75 / 81
    PREFILL_WAVES_BEHIND = (480, 2560, 3)
    # many workgroups and few keys: the tiled kernel reads a tile of keys once for 128 tokens and merges nothing (32 heads, 3 prompts
    # of 667, 2,016 workgroups: 27.5 / 30.8; 28 heads, 4 of 512, 1,792 24.4 / 26.5; 64 heads, 2 of 1,000 55.9 / 67.4; 40 heads of 64, 6 of
    # 130, 1,120 9.4 / 10.1)
    PREFILL_WAVES_MANY = ((1700, 1024), (1024, 256))                     # from so many workgroups on, with fewer keys
    # Waves of a workgroup, 8 / 4 / 2 (1, 2 or 4 workgroups a compute unit), us: 84 workgroups, 1,200 keys 12.5 / 14.4 / 22; 120 of 301
    # keys 8.5 / 7.8 / 9.4; 240 of 640 9.8 / 10.0 / 13.9; 512 of 40 14.6 / 8.8 / 7.5; 560 of 640 20.5 / 13.3 / 15.4; 640 of 301 (64 heads)
    # 19.4 / 14.2 / 10.7; 840 of 450 26 / 16.3 / 14.5; 812 of 901 29 / 20.5 / 20.5; 1,148 of 1,300 43 / 31.6 / 28.2; 1,792 of 2,048 76 /
    # 58 / 50
    PREFILL_WAVES = ((8, 256, 640), (4, 528, 65), (4, 576, 512), (4, 1024, 896), (4, 1400, 2560))    # waves, up to so many workgroups, from so many keys on
    PACKED_KEEPS_FREE = 0.3          # share of the device's memory that packed weight copies leave free
    PREFILL_F32_MIN_TOKENS = 32      # float32 steps with a portion of at least this many tokens go to the tiled float32 kernel
    # decode attention cuts the keys into runs so that about DECODE_WAVES waves are at work, with at most
    # DECODE_MAX_RUNS places for partial results per request and head. The kernel keeps two waves a SIMD (2,048 on
    # the chip); 1,536 is what the step likes best (1.5B shape, batch 32 and 64: 2.07 and 2.77 ms with 1,024, 2.02
    # and 2.71 with 1,536, 2.11 and 2.75 with 2,048; 7B shape, batch 160: 10.85, 10.05, 10.15 ms; batch 1 to 16 the same)
    DECODE_WAVES = 1536
    # where the same number of runs for every request leaves more than a fifth of those waves unused (1,024 pairs
    # of a request and a kv head: one run each), the requests of a decode step share one run length instead: the
    # shortest with which their runs together stay within DECODE_WAVES, so that a long request gets more runs than a
    # short one (256 requests on 4 kv heads, contexts of 1,050 to 3,150 keys: 263 -> 245 us a layer; contexts of one
    # length are cut as before). Everywhere else it is level or behind (32 requests: 30 -> 33 us).
    DECODE_SHARED_BELOW = 0.8
    DECODE_MAX_RUNS = 256
    # what a step's plan of attention is made by, beside its sizes
    ATTENTION_PLAN_RULES = ("PREFILL_PARTS", "PREFILL_WORKGROUPS", "PREFILL_WAVES_REACH", "PREFILL_WAVES_FEW", "PREFILL_WAVES_BEHIND",
                            "PREFILL_WAVES_MANY", "PREFILL_WAVES", "DECODE_WAVES", "DECODE_MAX_RUNS", "DECODE_SHARED_BELOW")
    # attention with mixed heads: from so many tokens a step on a workgroup takes 16 queries instead of 8 (fewer would
    # leave compute units without one)
    MIXED_WIDE_TOKENS = 6144
    # What a captured decode step of up to CHAIN_MAX_ROWS rows does between two layers' attention runs in one launch (`layer_chain.hip`),
    # for the widths that the kernel is built for and as far as K of the sums fits its registers. Measured in a captured graph, every
    # layer's weights from memory (us a layer, this / the six kernels, 1 and 8 rows): width 1,536, 8,960 hidden values 26.1 / 36.9 and
    # 33.1 / 39.8, 4,096 21.3 / 29.0 and 25.9 / 30.4; width 2,048, 11,008 35.3 / 46.2 and 42.0 / 49.5, 5,632 27.5 / 35.0 and 31.0 /
    # 37.3; width 1,024, 2,816 18.3 / 27.1 and 23.0 / 28.3, 8,192 20.4 / 30.6 and 26.7 / 32.0. Steps of the 1.5B shape: one request
    # 1,437 -> 1,145, 4 requests of 16,000 keys 1,791 -> 1,568, 8 of 2,048 1,572 -> 1,404. Steps that are launched kernel by kernel
    # keep their kernels. Values on their way between workgroups lie in memory that one fill prepares for CHAIN_CALLS layers.
    CHAIN_MAX_ROWS = 8
    CHAIN_WIDTHS = (1024, 1536, 2048)
    CHAIN_CALLS = 32
    CHAIN_WORKGROUPS = None          # workgroups of a launch (None: the compute units)
    CHAIN_PATIENCE = 256             # looks for values, about 1 us each, before a workgroup does what nobody has taken
    CHAIN_LIMIT = 1 << 14
    # the matrix-core attention kernels take heads up to 256; wider ones (a latent that all heads share) run on the
    # wave-per-token kernel, in either precision
    LARGEST_MATRIX_CORE_HEAD = 256
    LARGEST_HEAD = 1024

    def __init__(self, device="cuda:0", packed_weights=True) -> None:
        """`packed_weights` (True, False, or the roles that get one, as the parts name them in
        `prepare_linear`: "qkv", "attn_out", "gate_up", "down", "head"): keep a second copy of every bfloat16 weight in the order in which the
        matrix cores take it, for the products that run in passes over the weight or in tiles: decode, portions of prompts, and
        whole ones of thousands of tokens. It doubles the memory of the weights and makes those products 10-25 % faster, and it
        is what the fused epilogues (activation, rotation and cache write) work on; without it products of up to
        `SKINNY_MAX_ROWS` rows stream the weights as they are stored and larger ones go to the library."""
        self.device = torch.device(device)
        if isinstance(packed_weights, (bool, int)) or packed_weights is None:
            self.packed_weights = bool(packed_weights)
            self.packed_roles = None
        else:
            self.packed_roles = frozenset(packed_weights)
            self.packed_weights = bool(self.packed_roles)
        if self.device.type != "cuda" or not torch.cuda.is_available():
            raise KernelError("HipOps needs an AMD GPU (torch.cuda is not available): there is no CPU path")
        name = torch.cuda.get_device_properties(self.device).gcnArchName
        if not name.startswith("gfx950"):
            raise KernelError(f"the kernels are built for gfx950 (MI355X); this device is {name}")
        self._device_index = self.device.index if self.device.index is not None else torch.cuda.current_device()
        self._compute_units = torch.cuda.get_device_properties(self.device).multi_processor_count
        # (a device without a number is no tensor's device: `_own` refuses them one by one)
        self._owned = functools.partial(calls.native().owned, -1 if self.device.index is None else self.device.index)
        self._empty = functools.partial(calls.native().empty, self._device_index)       # (shape, dtype) -> tensor
        self._lib = None
        self._tuning = False
        self.library_timed_rows = self.library_timed_portion = 0
        self._packed_left_out = 0
        self._tile_plans: Dict[tuple, Optional[tuple]] = {}
        self._large_plans: Dict[tuple, object] = {}       # of `_tiled` and `_large_each`
        self._ops = ctypes.CDLL(str(build.ensure("ops")))
        self._declare()
        self._attn: Dict[int, ctypes.CDLL] = {}
        self._mixed: Dict[int, ctypes.CDLL] = {}
        # pinned staging buffers for `upload`, used in turn: [host tensor, its numpy view, event of the last copy]
        self._uploads = [[None, None, None] for _ in range(self.UPLOAD_BUFFERS)]
        self._next_upload = 0
        # what a kernel whose workgroups wait for one another writes if a wait came to its end (`raise_failures`)
        self._gave_up = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        self._gave_up_np = self._gave_up.numpy()

    # ------------------------------------------------------------ plumbing
    UPLOAD_BUFFERS = 8

    def upload(self, values: np.ndarray) -> torch.Tensor:
        """Through pinned memory, so that the copy is queued like a kernel: `torch.tensor(..., device=...)` copies
        from pageable memory and returns only when everything queued before it is done, which made the host
        wait for the running step three times per sampled step."""
        values = np.ascontiguousarray(values)
        dtype = torch.from_numpy(np.empty(0, dtype=values.dtype)).dtype
        nbytes = values.nbytes
        if nbytes == 0:
            return self._empty(values.shape, dtype)
        slot = self._uploads[self._next_upload]
        self._next_upload = (self._next_upload + 1) % len(self._uploads)
        if slot[2] is not None:
            slot[2].synchronize()                       # the copy made out of this buffer some calls ago is done
        if slot[0] is None or slot[0].numel() < nbytes:
            slot[0] = torch.empty(max(4096, 2 * nbytes), dtype=torch.uint8, pin_memory=True)
            slot[1] = slot[0].numpy()
            slot[2] = torch.cuda.Event()
        slot[1][:nbytes] = values.reshape(-1).view(np.uint8)
        dev = self._empty(nbytes, torch.uint8)
        dev.copy_(slot[0][:nbytes], non_blocking=True)
        slot[2].record()
        return dev.view(dtype).view(values.shape)

    def _declare(self) -> None:
        o = self._ops
        o.distie_scatter_i32.argtypes = [_P, _P, _P, _I, _L, _P]
        o.distie_clear_rows.argtypes = [_P, _I, _I, _P]
        o.distie_embed.argtypes = [_P, _P, _I, _P, _I, _I, _I, _F, _P]
        o.distie_rmsnorm.argtypes = [_P, _P, _I, _I, _P, _I, _P, _I, _I, _I, _F, _P]
        o.distie_rope_kv_write.argtypes = [_P, _I, _I, _P, _I, _P, _P, _P, _P, _P, _I, _P, _I, _I, _I, _I, _I, _I, _I, _P]
        o.distie_rope_table.argtypes = [_P, _P, _P, _I, _I, _P]
        o.distie_silu_mul.argtypes = [_P, _I, _I, _P, _I, _I, _I, _P]
        o.distie_sum_slices.argtypes = [_P, _I, _L, _P, _I, _P]
        o.distie_gather_rows.argtypes = [_P, _P, _P, _I, _L, _I, _P]
        o.distie_gemm_generic.argtypes = [_P, _I, _P, _I, _P, _P, _I, _I, _I, _I, _P]
        o.distie_gemv_rows.argtypes = [_P, _I, _P, _I, _P, _P, _I, _I, _I, _I, _P]
        o.distie_rows_f32_slices.argtypes = [_I, _I, _I, _I]
        o.distie_rows_f32_waves.argtypes = [_I, _I, _I, _I]
        o.distie_rows_f32.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _I, _F, _F, _F, _P]
        o.distie_rows_f32_rotary.argtypes = [_P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _P]
        o.distie_gemm_skinny_slices.argtypes = [_I, _I, _I]
        o.distie_gemm_skinny_bf16.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _P]
        o.distie_pack_rows.argtypes = [_P, _P, _P, _I, _I, _P]
        o.distie_gemm_packed_bf16.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _I, _F, _F, _F, _P]
        o.distie_gemm_packed_wide_bf16.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _F, _F, _F, _P]
        o.distie_gemm_packed_wide_slices.argtypes = [_I, _I]
        o.distie_gemm_packed_wide_qkv_bf16.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _P]
        o.distie_gemm_packed_rotary_bf16.argtypes = [_P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _P]
        o.distie_packed_tiles_plan.argtypes = [_I, _I, _I, _I, _I, _F] + 3 * [ctypes.POINTER(_I)]
        o.distie_packed_tiles_bf16.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _F, _F, _F, _P]
        o.distie_packed_tiles_rotary_bf16.argtypes = [_P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _I, _P]
        o.distie_large_tiles_plan.argtypes = [_I, _I, _I, _I, _I, _F] + 2 * [ctypes.POINTER(_I)] + [ctypes.POINTER(_F)]
        o.distie_large_tiles_grid.argtypes = [_I, _I, _I] + 2 * [ctypes.POINTER(_I)]
        o.distie_large_tiles_bf16.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _F, _F, _F, _P]
        o.distie_large_tiles_each_bf16.argtypes = [_P, _P, _P, _I, _I, _I, _P, _I, _P]
        o.distie_large_tiles_rotary_bf16.argtypes = [_P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _I, _P]
        o.distie_gemm_packed_each_bf16.argtypes = [_P, _P, _P, _I, _I, _I, _P, _P]
        o.distie_decode_norm_fits.argtypes = [_I]
        o.distie_decode_product_residual.argtypes = [_P, _P, _P, _P, _I, _I, _I, _P]
        o.distie_decode_norm_product.argtypes = [_P, _P, _F, _P, _P, _P, _I, _I, _I, _I, _P, _P, _P, _P,
                                                 _I, _I, _I, _I, _I, _P]
        o.distie_layer_chain_fits.argtypes = [_I, _I, _I, _I, _I, _I]
        o.distie_layer_chain_claims.argtypes = [_I]
        o.distie_layer_chain.argtypes = [_P, _P, _P, _P, _P, _F, _P, _P, _P, _P, _P, _F, _P, _P, _P, _P, _P, _P, _P] + 9 * [_I] + \
            [_P, _P, _I, _I, _I, _I, _P]
        o.distie_hyper_step.argtypes = [_P, _I, _P, _P, _I, _I, _P, _I, _L, _I, _P, _P, _P, _P, _I, _I, _F, _P, _I, _I, _I, _P]
        o.distie_causal_conv.argtypes = [_P, _I, _L, _P, _I, _I, _P, _P, _I, _L, _I, _P, _P, _P, _P, _I, _I, _P]
        o.distie_conv_state.argtypes = [_P, _I, _L, _I, _P, _P, _P, _I, _I, _I, _P]
        o.distie_conv_rope_kv_write.argtypes = [_P, _I, _L, _P, _I, _I, _P, _P, _I, _F, _P, _P, _P, _I, _P, _P, _P, _P,
                                                _I, _I, _I, _I, _I, _I, _I, _I, _I, _P, _F, _I, _P, _P, _F, _I, _I, _I, _P]
        o.distie_sigmoid_gate.argtypes = [_P, _I, _I, _I, _P, _I, _L, _P, _I, _I, _I, _P]
        o.distie_rmsnorm_gate.argtypes = [_P, _P, _I, _F, _P, _I, _L, _P, _I, _I, _I, _I, _I, _I, _P]
        o.distie_norm_chain.argtypes = [_P, _I, _I, _P, _P, _I, _I, _P, _F, _F, _P, _F, _P, _P, _F, _P, _I, _P, _I, _I, _P]
        o.distie_gated_decay_scan.argtypes = [_P, _I, _L, _P, _P, _L, _P, _P, _I, _P, _P, _P, _P, _I, _I, _I, _I, _F, _F, _P]
        o.distie_gated_decay_scan_chunked.argtypes = [_P, _I, _L, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _F, _F, _P]
        o.distie_lru_gates.argtypes = [_P, _I, _L, _P, _P, _P, _P, _I, _P, _F, _P, _P, _I, _I, _I, _P]
        o.distie_lru_scan.argtypes = [_P, _P, _P, _P, _I, _L, _I, _P, _I, _P, _P, _I, _I, _P]
        o.distie_lru_scan_chunked.argtypes = [_P, _P, _P, _P, _P, _P, _P, _I, _L, _I, _P, _I, _P, _P, _P, _I, _I, _I, _P]
        o.distie_route_topk.argtypes = [_P, _I, _P, _I, _P, _P, _P, _I, _I, _I, _I, _I, _P, _I, _I, _F, _I, _P]
        o.distie_route_glu.argtypes = [_P, _I, _L, _I, _P, _P, _I, _I, _I, _I, _F, _F, _F, _I, _I, _P, _I, _P]
        o.distie_route_topk_glu.argtypes = [_P, _P, _P, _I, _I, _P, _I, _L, _I, _I, _I, _I, _I, _F, _F, _F, _I, _P, _I, _I, _F, _I, _I, _P, _I, _P]
        o.distie_softcap_f32.argtypes = [_P, _L, _F, _P]
        o.distie_route_scale.argtypes = [_P, _I, _L, _P, _P, _I, _I, _I, _I, _P]
        o.distie_scale_f32.argtypes = [_P, _L, _F, _P]
        o.distie_activation.argtypes = [_P, _I, _I, _P, _I, _L, _I, _P]
        o.distie_decay_scan.argtypes = [_P, _I, _L, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _P, _I, _I, _F, _P]
        o.distie_decay_scan_chunked.argtypes = [_P, _I, _L, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _P, _I, _I, _F, _P]
        o.distie_delta_scan.argtypes = [_P, _I, _L, _P, _L, _P, _L, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _F, _F, _P]
        o.distie_delta_scan_chunked.argtypes = [_P, _I, _L, _P, _L, _P, _L, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P,
                                                _P, _I, _I, _I, _I, _I, _I, _F, _F, _P]
        o.distie_latent_norm_rope_write.argtypes = [_P, _I, _L, _I, _P, _I, _P, _F, _I, _P, _F, _I, _P, _I, _P, _P, _I, _P,
                                                    _I, _I, _I, _I, _P]
        o.distie_latent_queries.argtypes = [_P, _I, _I, _I, _P, _I, _P, _I, _I, _I, _I, _I, _I, _P, _F, _I, _P]
        o.distie_rope_heads.argtypes = [_P, _I, _I, _I, _P, _I, _I, _I, _I, _I, _P, _F, _I, _P]
        o.distie_heads_linear.argtypes = [_P, _I, _I, _P, _I, _P, _I, _I, _I, _I, _I, _P]
        o.distie_head_gate.argtypes = [_P, _I, _I, _I, _P, _I, _L, _P, _I, _I, _I, _P]
        o.distie_ssm_scan.argtypes = [_P, _I, _L, _P, _L, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _P]
        o.distie_ssm_scan_chunked.argtypes = [_P, _I, _L, _P, _L, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I,
                                              _I, _I, _P]
        o.distie_gate_rmsnorm.argtypes = [_P, _P, _I, _F, _P, _I, _L, _P, _I, _I, _I, _I, _I, _P]
        o.distie_glu_mul.argtypes = [_P, _I, _I, _P, _I, _I, _I, _I, _F, _F, _F, _P]
        o.distie_group_chain.argtypes = [_P, _I, _I, _P, _F, _I, _P, _P, _P, _P, _I, _P, _P, _I, _I, _I, _P, _I, _P, _P, _P]
        o.distie_token_shift.argtypes = [_P, _I, _P, _I, _P, _P, _P, _P, _P, _I, _I, _P]
        o.distie_wkv_scan.argtypes = [_P, _P, _P, _P, _I, _L, _P, _I, _L, _I, _P, _P, _P, _P, _P, _F, _P, _I, _P, _P, _I, _I,
                                      _I, _P]
        o.distie_wkv_scan_chunked.argtypes = [_P, _P, _P, _P, _I, _L, _P, _P, _P, _P, _F, _P, _I, _P, _P, _P, _P, _P, _I, _I, _I,
                                              _I, _P]
        o.distie_tanh_f32.argtypes = [_P, _L, _P, _I, _I, _P]
        o.distie_mixed_attention_generic.argtypes = [_P, _I, _L, _P, _P, _I, _P, _P, _P, _I, _P, _P, _I, _I, _I, _I, _I, _F,
                                                     _I, _I, _F, _P, _I, _P, _P, _P]
        o.distie_argmax.argtypes = [_P, _P, _I, _I, _P, _P, _P]
        o.distie_argmax_parts.argtypes = [_I, _I]
        o.distie_sample.argtypes = [_P, _P, _P, _P, _P, _I, _I, _P, _P, _P, _P]
        calls.quicken(o)

    def tune_library_products(self, on: bool) -> None:
        """While on, every new shape of a large product has the library's candidate kernels timed, and the
        fastest is kept for that shape, and for the other row counts of its class of 32 rows, from then on; shapes
        first met while off take their class's choice, or the library's first. Products of up to `PACKED_MAX_ROWS`
        rows do not go to the library at all (`PACKED_MAX_ROWS_EAGER` outside captured steps; large weights:
        see there). The caller that has had every class up to some number of rows timed says so in
        `library_timed_rows`: up to there large weights with more rows than K leave the packed kernels at 65 rows."""
        self._tuning = bool(on)

    def graphs_supported(self) -> bool:
        """Every kernel launches on torch's current stream and keeps its scratch at fixed
        addresses, so a step can be captured into a HIP graph."""
        return True

    def _stream(self):
        # torch's current stream as a raw handle; the direct getter saves the 4 us a call that building a
        # Stream object costs (a step makes some 200 calls)
        if _raw_stream is not None:
            return _raw_stream(self._device_index)
        return torch.cuda.current_stream(self.device).cuda_stream

    def attention_library(self, head_dim: int) -> ctypes.CDLL:
        lib = self._attn.get(head_dim)
        if lib is None:
            if head_dim % 2 or not 2 <= head_dim <= self.LARGEST_HEAD:
                raise KernelError(f"attention kernels take even head sizes up to {self.LARGEST_HEAD}, not {head_dim}")
            lib = ctypes.CDLL(str(build.ensure(f"attn_d{head_dim}")))
            lib.distie_attention_generic.argtypes = [_P, _I, _L, _P, _P, _I, _P, _P, _P, _I, _P, _P,
                                                     _I, _I, _I, _I, _F, _I, _P, _F, _P, _P, _P, _I, _I, _I, _P]
            lib.distie_attention_columns_f32_runs.argtypes = [_I, _I, _I, _I, _I, _L, _I]
            lib.distie_attention_columns_f32_pays.argtypes = [_I, _I, _I, _I, _I, _I, _I]
            lib.distie_attention_columns_f32.argtypes = [_P, _L, _P, _P, _P, _P, _P, _I, _P, _P, _I, _I, _I, _I, _I, _F, _I,
                                                         _P, _P, _P, _I, _P]
            lib.distie_attention_f32_plan.argtypes = [_I, _I, _I, _I, ctypes.POINTER(_I), ctypes.POINTER(_I)]
            lib.distie_attention_prefill_bf16.argtypes = [_P, _L, _P, _P, _P, _P, _P, _I, _P, _P, _I, _I, _I, _I, _I,
                                                          _F, _I, _I, _P, _P, _P, _I, _P, _P]
            lib.distie_attention_prefill_f32.argtypes = lib.distie_attention_prefill_bf16.argtypes
            lib.distie_attention_prefill_keys.argtypes = [_P, _L, _P, _P, _P, _P, _P, _I, _P, _P, _I, _I, _I, _I, _I, _F, _I, _I,
                                                          _P, _I, _P]
            lib.distie_attention_decode_bf16.argtypes = [_P, _L, _P, _P, _P, _P, _P, _I, _P, _P, _P, _P, _I, _I, _I,
                                                         _I, _F, _I, _I, _I, _I, _P, _P, _I, _P]
            lib.distie_attention_decode_together.argtypes = [_I, _I, _I]
            lib.distie_attention_decode_run_len.argtypes = [_P, _I, _I, _I, _P, _P]
            if lib.distie_attention_head_dim() != head_dim:
                raise KernelError("attention library was built for another head size")
            calls.quicken(lib)
            self._attn[head_dim] = lib
        return lib

    def mixed_attention_library(self, head_dim: int) -> ctypes.CDLL:
        lib = self._mixed.get(head_dim)
        if lib is None:
            lib = ctypes.CDLL(str(build.ensure(f"mixattn_d{head_dim}")))
            lib.distie_mixed_fits.argtypes = [_I, _I]
            lib.distie_mixed_attention_bf16.argtypes = [_P, _L, _P, _P, _P, _P, _P, _I, _P, _P, _I, _I, _I, _I, _I, _F, _I, _I,
                                                        _F, _P, _I, _P, _P, _I, _I, _I, _I, _P, _P, _P]
            if lib.distie_mixed_head_dim() != head_dim:
                raise KernelError("the library of attention with mixed heads was built for another head size")
            calls.quicken(lib)
            self._mixed[head_dim] = lib
        return lib

    # (the constructor puts the native ones in their place)
    def _empty(self, shape, dtype):
        return torch.empty(shape, dtype=dtype, device=self.device)

    def _owned(self, *tensors) -> bool:
        return False

    def _own(self, *tensors) -> None:
        if self._owned(*tensors):
            return
        for t in tensors:
            if t is None:
                continue
            if t.device != self.device:
                raise KernelError(f"tensor on {t.device}, kernels run on {self.device}")
            if not t.is_contiguous():
                raise KernelError("kernels take contiguous tensors")

    @staticmethod
    def _check_cache(k_cache, v_cache, kv_heads, block_size, head_dim) -> None:
        if tuple(k_cache.shape[1:]) != (kv_heads, block_size, head_dim) or \
                tuple(v_cache.shape[1:]) != (kv_heads, head_dim, block_size) or k_cache.shape[0] != v_cache.shape[0]:
            raise KernelError("cache is not k [pages, kv_heads, block_size, head_dim], "
                              "v [pages, kv_heads, head_dim, block_size]")

    # ------------------------------------------------------------ operations
    def scatter_int32(self, table, index, value):
        self._own(table, index, value)
        if table.dtype != torch.int32 or index.dtype != torch.int32 or value.dtype != torch.int32 or \
                index.shape != value.shape:
            raise KernelError("scatter_int32 takes int32 tensors, one value for each index")
        _check(self._ops.distie_scatter_i32(table, index, value, index.numel(),
                                            table.numel(), self._stream()), "scatter_i32")
        _mark_written(table)

    def row_clearer(self, tensors):
        pieces, others, most = [], [], self._ops.distie_clear_rows_bytes()
        for t in tensors:
            self._own(t)
            size = t[0].numel() * t.element_size() if t.shape[0] else 0
            if size % 4 or t.data_ptr() % 4:
                others.append(t)
                continue
            pieces += [(t.data_ptr(), size, at, min(most, size - at)) for at in range(0, size, most)]
        held, rows = list(tensors), min((t.shape[0] for t in tensors), default=0)      # (kept while the table names them)
        table = torch.tensor(pieces, dtype=torch.int64).to(self.device) if pieces else None

        def clear(row: int) -> None:
            if held and not 0 <= row < rows:
                raise KernelError(f"there is no row {row} to clear")
            if table is not None:
                _check(self._ops.distie_clear_rows(table, len(pieces), row, self._stream()), "clear_rows")
            for t in others:
                t[row].zero_()
        return clear

    def embed(self, ids, table, scale=1.0):
        self._own(ids, table)
        out = self._empty((ids.shape[0], table.shape[1]), torch.float32)
        _check(self._ops.distie_embed(ids, table, _code(table), out,
                                      ids.shape[0], table.shape[1], table.shape[0], float(scale), self._stream()), "embed")
        return out

    def _norm_later(self, residual, weight, out_dtype) -> bool:
        """The norm of these rows can be left to the product that reads it."""
        return (self.packed_weights and self._fused(residual.shape[0]) and out_dtype == torch.bfloat16 and
                residual.dtype == torch.float32 and residual.dim() == 2 and
                weight.dtype in _CODES and bool(self._ops.distie_decode_norm_fits(residual.shape[1])))

    def _fused(self, rows: int) -> bool:
        return rows <= self.FUSED_MAX_ROWS and (self.FUSED_IN_CAPTURED_STEPS or not self.captured)

    def rmsnorm(self, x, weight, eps, out_dtype):
        self._own(x, weight)
        if x.dtype != torch.float32:
            raise KernelError("rmsnorm reads the float32 residual stream")
        if self._norm_later(x, weight, out_dtype):
            return PendingNorm(x, weight, eps, out_dtype)
        return self._rmsnorm_now(x, weight, eps, out_dtype)

    def _rmsnorm_now(self, x, weight, eps, out_dtype):
        out = self._empty(x.shape, out_dtype)
        _check(self._ops.distie_rmsnorm(x, None, _F32, 1, weight, _code(weight),
                                        out, _CODES[out_dtype], x.shape[0], x.shape[1], eps,
                                        self._stream()), "rmsnorm")
        return out

    def add_rmsnorm(self, residual, delta, weight, eps, out_dtype):
        if isinstance(delta, PendingProduct):
            self._own(residual, weight)
            if residual.dtype != torch.float32 or residual.shape != delta.shape:
                raise KernelError("add_rmsnorm: residual must be float32 and shaped like delta")
            # the product adds itself to the stream; what is left is the norm of the stream
            self._product_into_residual(delta, residual)
            return self.rmsnorm(residual, weight, eps, out_dtype)
        slices = 1
        delta = self.dense(delta) if isinstance(delta, PendingNorm) else delta
        if isinstance(delta, PartialSums):
            slices, delta = delta.slices, delta.data
        self._own(residual, delta, weight)
        if residual.dtype != torch.float32 or residual.shape != delta.shape[-2:]:
            raise KernelError("add_rmsnorm: residual must be float32 and shaped like delta")
        out = self._empty(residual.shape, out_dtype)
        _check(self._ops.distie_rmsnorm(residual, delta, _code(delta), slices,
                                        weight, _code(weight), out, _CODES[out_dtype],
                                        residual.shape[0], residual.shape[1], eps, self._stream()), "add_rmsnorm")
        _mark_written(residual)
        return out

    def _product_into_residual(self, product: PendingProduct, residual: torch.Tensor) -> None:
        x, weight, bias = product.x, product.weight, product.bias
        packed = getattr(weight, "_distie_packed")
        M, K = x.shape
        N = weight.shape[0]
        if packed.numel() != self._packed_elements(N, K, False):
            raise KernelError("linear: the packed copy does not belong to this weight")
        _check(self._ops.distie_decode_product_residual(
            x, packed, bias, residual,
            M, N, K, self._stream()), "decode_product_residual")
        _mark_written(residual)

    def raise_failures(self):
        if self._gave_up_np[0]:
            self._gave_up_np[0] = 0
            raise KernelError("layer_chain: a workgroup waited in vain for another one's values; what the steps since the last "
                              "look computed is void")

    # ---- a layer's end and the next one's beginning in one launch
    def _chain_fits(self, M, C, KO, inter, N) -> bool:
        return bool(self._ops.distie_layer_chain_fits(M, C, KO, inter, N, self._compute_units))

    def layer_tail(self, meta, residual, mixed, out_weight, norm_weight, eps, gate_up_weight, down_weight):
        if not self.captured or residual.dim() != 2 or residual.shape[0] > self.CHAIN_MAX_ROWS or \
                residual.shape[1] not in self.CHAIN_WIDTHS or mixed.dtype != torch.bfloat16 or residual.dtype != torch.float32:
            return None
        out_packed, gated, down_packed = (getattr(out_weight, "_distie_packed", None), getattr(gate_up_weight, "_distie_gated", None),
                                          getattr(down_weight, "_distie_packed", None))
        if out_packed is None or gated is None or down_packed is None:
            return None
        M, C = residual.shape
        KO, inter = mixed.shape[1], down_weight.shape[1]
        if mixed.shape[0] != M or tuple(out_weight.shape) != (C, KO) or tuple(gate_up_weight.shape) != (2 * inter, C) or \
                down_weight.shape[0] != C or norm_weight.dtype not in _CODES or tuple(norm_weight.shape) != (C,) or \
                out_packed.numel() != self._packed_elements(C, KO, False) or \
                gated.numel() != self._packed_elements(2 * inter, C, True) or \
                down_packed.numel() != self._packed_elements(C, inter, False) or not self._chain_fits(M, C, KO, inter, 0) or \
                residual.data_ptr() % 16 or mixed.data_ptr() % 16:
            return None
        self._own(residual, mixed, norm_weight)
        return LayerTail(self, residual, mixed, out_weight, norm_weight, eps, gate_up_weight, down_weight,
                         self._chain_buffers(meta, M, C, inter))

    def _chain_buffers(self, meta, M, C, inter):
        """int32 words of one launch, every byte 0xff: `mid`, `out` [M, C], `hidden` [M, inter] / 2, the claims. The launches of a
        step share a fill (each has words of its own)."""
        words = 2 * M * C + -(-M * inter // 8) * 4 + self._ops.distie_layer_chain_claims(self._compute_units)
        key = ("layer_chain", words)
        left = meta.scratch.get(key)
        if left is None or not left.shape[0]:
            left = torch.full((self.CHAIN_CALLS, -(-words // 64) * 64), -1, dtype=torch.int32, device=self.device)
        meta.scratch[key] = left[1:]
        return left[0]

    def _layer_chain(self, tail, following):
        """-> (new residual, q/k/v of the layer behind or None)"""
        M, C = tail.residual.shape
        KO, inter = tail._inner()
        out_weight, gate_up_weight, down_weight = tail.weights
        words = tail.scratch
        mid, out, hidden = words[:M * C], words[M * C:2 * M * C], words[2 * M * C:]
        claims = words[words.shape[0] - self._ops.distie_layer_chain_claims(self._compute_units):]
        norm_weight, eps = tail.norm
        qkv, rest, next_norm, next_eps, packed, bias = None, (None, None, None, None, 0, 0, 0, 0, 0), None, 0.0, None, None
        if following is not None:
            next_norm, next_eps, packed, bias, table, slots, k_cache, v_cache, heads, kv_heads, dim, block_size, write = following
            next_norm = self._f32(next_norm)
            qkv = self._empty((M, (heads + 2 * kv_heads) * dim), torch.bfloat16)
            rest = (table, slots, k_cache, v_cache, heads, kv_heads, dim, block_size, write)
        _check(self._ops.distie_layer_chain(
            tail.mixed, out_weight._distie_packed, tail.residual, mid,
            self._f32(norm_weight), eps, gate_up_weight._distie_gated, hidden,
            down_weight._distie_packed, out, next_norm, next_eps, packed, bias, qkv, *rest,
            M, C, KO, inter, claims, self._gave_up, self._compute_units, self.CHAIN_WORKGROUPS or self._compute_units,
            self.CHAIN_PATIENCE, self.CHAIN_LIMIT, self._stream()), "layer_chain")
        return out.view(torch.float32).view(M, C), qkv

    def dense(self, x):
        """The finished tensor of a value that an operation here returned in a form of its own (partial sums,
        a norm or a product that was left for later); any other tensor as it is."""
        if isinstance(x, PendingNorm):
            x.check()
            return self._rmsnorm_now(x.residual, x.weight, x.eps, x.dtype)
        if isinstance(x, PendingProduct):
            return self._linear(x.x, x.weight, x.bias, x.dtype, lazy=False)
        if isinstance(x, NormedSum):
            return self._norm_chain(x.terms, x.weights, x.eps, x.scale, None, None, None, None)
        if not isinstance(x, PartialSums):
            return x
        out = self._empty(tuple(x.shape), x.dtype)
        _check(self._ops.distie_sum_slices(x.data, x.slices, out.numel(), out,
                                           _CODES[x.dtype], self._stream()), "sum_slices")
        return out

    # ---- packed copies of weights: tiles of 16 rows x 32 k in the matrix cores' lane order
    @staticmethod
    def _row_map(N, gated, rotary):
        """Which row of the weight sits at each place of the packed copy's row blocks (-1: zeros)."""
        if gated:
            inter = N // 2
            j = torch.arange(-(-inter // 8) * 8, dtype=torch.int64).view(-1, 8)
            gate = torch.where(j < inter, j, -1)
            up = torch.where(j < inter, j + inter, -1)
            return torch.cat([gate, up], dim=1).reshape(-1)
        if rotary is not None:
            heads, kv_heads, dim = rotary
            lo = torch.arange(dim // 2, dtype=torch.int64).view(-1, 8)                 # [dim/16, 8]
            one = torch.cat([lo, lo + dim // 2], dim=1).reshape(-1)                   # rows of a q or k head
            turned = (torch.arange(heads + kv_heads, dtype=torch.int64)[:, None] * dim + one[None, :]).reshape(-1)
            return torch.cat([turned, torch.arange((heads + kv_heads) * dim, N, dtype=torch.int64)])
        rows = torch.full((-(-N // 16) * 16,), -1, dtype=torch.int64)
        rows[:N] = torch.arange(N)
        return rows

    @staticmethod
    def _packed_elements(N, K, gated):
        row_blocks = -(-(N // 2) // 8) if gated else -(-N // 16)
        return row_blocks * -(-K // 32) * 512

    def prepare_linear(self, weight, gated=False, rotary=None, role=None):
        if self.packed_roles is not None and role not in self.packed_roles:
            return
        if not self.packed_weights or weight.dtype != torch.bfloat16 or weight.dim() != 2 or weight.shape[1] % 8:
            return
        N, K = weight.shape
        name = "_distie_packed"
        if gated:
            if N % 2:
                return
            name = "_distie_gated"
        elif rotary is not None:
            heads, kv_heads, dim = rotary
            if dim % 16 or N != (heads + 2 * kv_heads) * dim:
                rotary = None                 # the fused kernel does not take it: the plain copy serves
            else:
                name = "_distie_rotary"
        if hasattr(weight, name):
            return
        self._own(weight)
        row_map = self._row_map(N, gated, rotary)
        if row_map.numel() % 16 or int(row_map.max()) >= N or int(row_map.min()) < -1 or \
                row_map.numel() // 16 * -(-K // 32) * 512 != self._packed_elements(N, K, gated):
            raise KernelError("prepare_linear: bad row map")
        # The copies are for speed, the cache is needed: a copy that would leave less than PACKED_KEEPS_FREE of the
        # card's memory free is left out (the product then streams the stored layout), said once.
        free, total = torch.cuda.mem_get_info(self.device)
        if free - 2 * self._packed_elements(N, K, gated) < self.PACKED_KEEPS_FREE * total:
            if not self._packed_left_out:
                _log.warning("packed weight copies are left out from here on: less than %.0f %% of the device's "
                             "memory would stay free", 100 * self.PACKED_KEEPS_FREE)
            self._packed_left_out += 1
            return
        row_map = row_map.to(device=self.device, dtype=torch.int32)
        packed = self._empty(self._packed_elements(N, K, gated), torch.bfloat16)
        _check(self._ops.distie_pack_rows(weight, packed, row_map,
                                          row_map.numel() // 16, K, self._stream()), "pack_rows")
        torch.cuda.current_stream(self.device).synchronize()      # row_map is freed on return
        # the copy lives and dies with the weight
        weight._distie_role = role
        setattr(weight, name, (packed, tuple(rotary)) if name == "_distie_rotary" else packed)

    def _norm_product(self, x: PendingNorm, packed, bias, out, mode, N, rotary=None):
        """`out` = the product of rmsnorm(x.residual) with the weight whose packed copy is `packed`, the norm
        computed inside the product."""
        x.check()
        M, K = x.shape
        table = slots = k_cache = v_cache = None
        heads = kv_heads = dim = block_size = write = 0
        if rotary is not None:
            table, slots, k_cache, v_cache, heads, kv_heads, dim, block_size, write = rotary
        norm_weight = x.weight
        if norm_weight.dtype != torch.float32:
            # the kernel takes the norm's weights in float32 (a bfloat16 value is one exactly); kept on the tensor
            norm_weight = getattr(x.weight, "_distie_f32", None)
            if norm_weight is None:
                norm_weight = x.weight._distie_f32 = x.weight.float()
        _check(self._ops.distie_decode_norm_product(
            x.residual, norm_weight, x.eps, packed, bias,
            out, mode, M, N, K, table, slots, k_cache, v_cache, heads, kv_heads, dim,
            block_size, write, self._stream()), "decode_norm_product")
        return out

    def linear_silu_mul(self, x, gate_up_weight):
        return self.linear_glu(x, gate_up_weight, "silu")

    def linear_glu(self, x, gate_up_weight, kind):
        """The gated product with the activation in its epilogue, on the GATED copy of the weight (steps of few rows);
        else the product, then `glu_mul`."""
        if kind not in self.ACTIVATIONS:
            raise KernelError(f"linear_glu: no activation named {kind!r}")
        return self._linear_gated(x, gate_up_weight, 1 if kind == "silu" else 1 | ((self.ACTIVATIONS[kind] + 1) << 8),
                                  lambda product: self.glu_mul(product, kind))

    CLAMPED = 5                      # the clamped activation, as the packed products number what stands on the gate

    def linear_clamped_glu(self, x, gate_up_weight, limit, slope, up_shift):
        if not limit > 0:
            raise KernelError("linear_clamped_glu: the limit must be positive")
        return self._linear_gated(self.dense(x), gate_up_weight, 1 | (self.CLAMPED << 8),
                                  lambda product: self.clamped_glu(product, limit, slope, up_shift),
                                  (float(limit), float(slope), float(up_shift)))

    def _linear_gated(self, x, gate_up_weight, gated, apart, clamp=(0.0, 1.0, 0.0)):
        """`gated`: 1, and above the low eight bits what stands on the gate; `apart`: the same on a finished product."""
        packed = getattr(gate_up_weight, "_distie_gated", None)
        if isinstance(x, PendingNorm) and packed is not None and gate_up_weight.shape[1] == x.shape[1]:
            N, K = gate_up_weight.shape
            if packed.numel() != self._packed_elements(N, K, True):
                raise KernelError("linear_silu_mul: the packed copy does not belong to this weight")
            out = self._empty((x.shape[0], N // 2), torch.bfloat16)
            return self._norm_product(x, packed, None, out, gated, N)
        x = self.dense(x)
        M, K = x.shape
        N = gate_up_weight.shape[0]
        if x.dtype == torch.float32 and gate_up_weight.dtype == torch.float32 and gate_up_weight.shape[1] == K and N % 2 == 0 and \
                N * K >= self.ROWS_F32_MIN_ELEMENTS and self._ops.distie_rows_f32_slices(M, N, K, 1):
            self._own(x, gate_up_weight)
            out = self._empty((M, N // 2), torch.float32)
            _check(self._ops.distie_rows_f32(x, gate_up_weight, None, out, M, N, K, gated, 1,
                                             *clamp, self._stream()), "rows_f32")
            return out
        plan, large = None, False
        if packed is not None and x.dtype == torch.bfloat16:
            plan, large = self._tiled(x.shape[0], *gate_up_weight.shape, "gated", (x,))
        if packed is None or x.dtype != torch.bfloat16 or \
                (plan is None and x.shape[0] > self._packed_rows(x.shape[0], *gate_up_weight.shape)):
            return apart(self.linear(x, gate_up_weight))
        self._own(x)
        if gate_up_weight.shape[1] != K:
            raise KernelError(f"linear: x is [{M}, {K}], weight is {list(gate_up_weight.shape)}")
        if packed.numel() != self._packed_elements(N, K, True):
            raise KernelError("linear_silu_mul: the packed copy does not belong to this weight")
        if plan is not None:
            return self._run_tiles(plan, x, packed, None, x.dtype, M, N, K, gated, clamp=clamp, large=large)
        out = self._empty((M, N // 2), x.dtype)
        if M <= self.ONE_WAVE_MAX_ROWS:
            _check(self._ops.distie_gemm_packed_bf16(x, packed, None, out, _code(out),
                                                     M, N, K, gated, *clamp, self._stream()), "gemm_packed_bf16")
        else:
            _check(self._ops.distie_gemm_packed_wide_bf16(
                x, packed, None, out, _code(out), M, N, K, gated,
                self._pass_blocks(M, N * K), *clamp, self._stream()), "gemm_packed_wide_bf16")
        return out

    def linear_rope_kv_write(self, x, weight, bias, meta, group, k_cache, v_cache, inv_freq, num_heads, num_kv_heads,
                             head_dim, write):
        held = getattr(weight, "_distie_rotary", None)
        if isinstance(x, PendingNorm) and held is not None and held[1] == (num_heads, num_kv_heads, head_dim) and \
                inv_freq is not None and 2 * inv_freq.shape[0] == head_dim and k_cache.dtype == torch.bfloat16 and \
                weight.shape[1] == x.shape[1]:
            packed = held[0]
            slots = meta.groups[group].slots
            self._own(bias, k_cache, v_cache, inv_freq, slots)
            M, K = x.shape
            N = weight.shape[0]
            if N != (num_heads + 2 * num_kv_heads) * head_dim:
                raise KernelError(f"linear: weight is {list(weight.shape)} for {num_heads} + 2 x {num_kv_heads} heads")
            if bias is not None and (bias.dtype != torch.float32 or bias.shape[0] != N):
                raise KernelError("linear: bias must be float32 [N]")
            if packed.numel() != self._packed_elements(N, K, False):
                raise KernelError("linear_rope_kv_write: the packed copy does not belong to this weight")
            self._check_cache(k_cache, v_cache, num_kv_heads, meta.block_size, head_dim)
            if M != meta.num_tokens or slots.shape[0] != M:
                raise KernelError("linear_rope_kv_write: rows do not match the batch")
            table = self._rope_table(meta, inv_freq)
            out = self._empty((M, N), torch.bfloat16)
            return self._norm_product(x, packed, bias, out, 2, N, rotary=(
                table, slots, k_cache, v_cache, num_heads, num_kv_heads, head_dim, meta.block_size, 1 if write else 0))
        x = self.dense(x)
        M, K = x.shape
        N = weight.shape[0]
        if x.dtype == torch.float32 and weight.dtype == torch.float32 and k_cache.dtype == torch.float32 and \
                inv_freq is not None and 2 * inv_freq.shape[0] == head_dim and head_dim % 16 == 0 and \
                N == (num_heads + 2 * num_kv_heads) * head_dim and weight.shape[1] == K and \
                (bias is None or (bias.dtype == torch.float32 and bias.shape[0] == N)) and \
                N * K >= self.ROWS_F32_MIN_ELEMENTS and self._ops.distie_rows_f32_slices(M, N, K, 1):
            slots = meta.groups[group].slots
            self._own(x, weight, bias, k_cache, v_cache, inv_freq, slots)
            self._check_cache(k_cache, v_cache, num_kv_heads, meta.block_size, head_dim)
            if M != meta.num_tokens or slots.shape[0] != M:
                raise KernelError("linear_rope_kv_write: rows do not match the batch")
            table = self._rope_table(meta, inv_freq)
            out = self._empty((M, N), torch.float32)
            _check(self._ops.distie_rows_f32_rotary(
                x, weight, bias, out,
                table, slots, k_cache, v_cache, M, K, num_heads, num_kv_heads,
                head_dim, meta.block_size, 1 if write else 0, self._stream()), "rows_f32_rotary")
            return out
        plan, large = None, False
        fused = held is not None and held[1] == (num_heads, num_kv_heads, head_dim) and x.dtype == torch.bfloat16 and \
            inv_freq is not None and 2 * inv_freq.shape[0] == head_dim and k_cache.dtype == torch.bfloat16
        if fused:
            plan, large = self._tiled(x.shape[0], *weight.shape, "rotary", (x, bias, k_cache))
            fused = plan is not None or x.shape[0] <= self._packed_rows(x.shape[0], *weight.shape)
        if not fused:
            return self.rope_kv_write(self.linear(x, weight, bias), meta, group, k_cache, v_cache, inv_freq,
                                      num_heads, num_kv_heads, head_dim, write)
        packed = held[0]
        slots = meta.groups[group].slots
        self._own(x, bias, k_cache, v_cache, inv_freq, slots)
        M, K = x.shape
        N = weight.shape[0]
        if weight.shape[1] != K or N != (num_heads + 2 * num_kv_heads) * head_dim:
            raise KernelError(f"linear: x is [{M}, {K}], weight is {list(weight.shape)}")
        if bias is not None and (bias.dtype != torch.float32 or bias.shape[0] != N):
            raise KernelError("linear: bias must be float32 [N]")
        if packed.numel() != self._packed_elements(N, K, False):
            raise KernelError("linear_rope_kv_write: the packed copy does not belong to this weight")
        self._check_cache(k_cache, v_cache, num_kv_heads, meta.block_size, head_dim)
        if M != meta.num_tokens or slots.shape[0] != M:
            raise KernelError("linear_rope_kv_write: rows do not match the batch")
        if plan is None and M >= self.WIDE_QKV_MIN_ROWS and N * K > self.ROW_GROUPS_MAX_ELEMENTS:
            # more than one group of 16 rows against a weight that fills the chip through the wide kernel: the
            # epilogue kernel would read the weight once per group, so the product runs wide (weights once, K in
            # slices) and the rotation with the cache write behind it adds the slices
            slices = self._ops.distie_gemm_packed_wide_slices(N, K)
            shape, dtype = ((M, N), torch.bfloat16) if slices == 1 else ((slices, M, N), torch.float32)
            product = self._empty(shape, dtype)
            _check(self._ops.distie_gemm_packed_wide_qkv_bf16(
                x, packed, bias, product,
                _code(product), M, K, num_heads, num_kv_heads, head_dim, self._pass_blocks(M, N * K), self._stream()),
                "gemm_packed_wide_qkv_bf16")
            if slices > 1:
                product = PartialSums(product, torch.bfloat16)
            return self.rope_kv_write(product, meta, group, k_cache, v_cache, inv_freq, num_heads, num_kv_heads,
                                      head_dim, write)
        table = self._rope_table(meta, inv_freq)
        out = self._empty((M, N), torch.bfloat16)
        if plan is not None:
            kernel, name = (self._ops.distie_large_tiles_rotary_bf16, "large_tiles_rotary_bf16") if large else \
                (self._ops.distie_packed_tiles_rotary_bf16, "packed_tiles_rotary_bf16")
            _check(kernel(
                x, packed, bias, out,
                table, slots, k_cache, v_cache, M, K, num_heads,
                num_kv_heads, head_dim, meta.block_size, 1 if write else 0, plan[0], self._stream()), name)
            return out
        _check(self._ops.distie_gemm_packed_rotary_bf16(
            x, packed, bias, out,
            table, slots, k_cache, v_cache, M, K, num_heads,
            num_kv_heads, head_dim, meta.block_size, 1 if write else 0, self._stream()), "gemm_packed_rotary_bf16")
        return out

    def _packed_rows(self, M: int, N: int, K: int) -> int:
        """Most rows of x that go through the kernels on the packed copy of an [N, K] weight, for a product of M rows."""
        if N * K > self.PACKED_LARGE_ELEMENTS:
            if K > N:
                return self.PACKED_MAX_ROWS_LARGE
            return self.PACKED_MAX_ROWS_LARGE_WIDE_TIMED if M <= self.library_timed_rows else self.PACKED_MAX_ROWS_LARGE_WIDE
        return self.PACKED_MAX_ROWS if self.captured else self.PACKED_MAX_ROWS_EAGER

    TILE_PLANS = 4096                # products whose cut is remembered

    def _tiles(self, M: int, N: int, K: int, kind: str, cut_us: Optional[float] = None):
        """(shape, slices) of the tiled kernels for a product of M rows with an [N, K] weight, None if another kernel is
        the better one. kind: "plain", "gated" or "rotary"; cut_us: what a cut of K costs the reader of the result beyond
        reading the slices (None: it must not be cut)."""
        if M < self.TILES_MIN_ROWS:
            return None
        key = (M, N, K, kind, cut_us, self.captured, self.library_timed_rows, self.library_timed_portion)
        try:
            return self._tile_plans[key]
        except KeyError:
            pass
        plan = None
        shape, slices, workgroups = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int(0)
        if self._ops.distie_packed_tiles_plan(M, N, K, kind == "gated", cut_us is not None, cut_us or 0.0, ctypes.byref(shape),
                                              ctypes.byref(slices), ctypes.byref(workgroups)) and \
                self._tiles_take(M, N, K, kind, shape.value, slices.value, workgroups.value):
            plan = (shape.value, slices.value)
        if len(self._tile_plans) >= self.TILE_PLANS:
            self._tile_plans.clear()
        self._tile_plans[key] = plan
        return plan

    def _tiles_take(self, M, N, K, kind, shape, slices, workgroups) -> bool:
        """Whether a product of the plan (shape, slices) and so many workgroups is to run in tiles: see the constants."""
        elements, work = N * K, M * N * K
        # whether the library's kernels for these rows were chosen by timing (it goes by classes of 32 rows)
        timed = M <= self.library_timed_rows or -(-M // 32) == -(-self.library_timed_portion // 32)
        passes = self._packed_rows(M, N, K)               # rows of x up to which the passes over a packed copy go
        one_round = workgroups <= self._compute_units
        small = elements <= self.ROW_GROUPS_MAX_ELEMENTS
        if not self.captured and M <= self.TILES_HOST_ROWS and elements <= self.TILES_SMALL_GATED and \
                (M >= self.TILES_MIN_ROTARY_ROWS or kind == "plain") and \
                work <= (self.TILES_LEVEL_GATED_WORK if kind == "gated" else self.TILES_MAX_WORK):
            return True
        if kind == "rotary":
            return M >= self.TILES_MIN_ROTARY_ROWS and (M > passes or not small) and one_round and work <= self.TILES_MAX_WORK and \
                (shape == 0 or (shape == 1 and elements > self.TILES_LARGE_ROTARY and not timed))
        if kind == "gated":
            if small:
                return M > passes and work <= self.TILES_MAX_SMALL_GATED_WORK
            if elements <= self.TILES_SMALL_GATED:
                return (M > passes or (M > 80 and one_round)) and work <= self.TILES_MAX_SMALL_GATED_WORK
            level = M <= self.PACKED_MAX_ROWS or not self.captured
            return work <= (self.TILES_LEVEL_GATED_WORK if level else self.TILES_MAX_GATED_WORK)
        long = K >= 2 * N
        if not long and work > self.TILES_MAX_WORK:
            return False
        if slices == 1:
            return one_round and not (long and M > self.TILES_LONG_ROWS) and \
                (shape <= 1 or (shape == 2 and N > K and not small and not timed))
        if elements <= self.TILES_SMALL_ELEMENTS:
            return self.PACKED_MAX_ROWS < M <= self.TILES_LONG_ROWS and not timed
        if M < self.TILES_CUT_ROWS:
            return elements <= self.PACKED_LARGE_ELEMENTS // 2 and N <= self.TILES_FEW_WEIGHT_ROWS
        if M <= 80 and elements > self.PACKED_LARGE_ELEMENTS:
            return one_round and shape == 0
        if long and M > self.TILES_LONG_ROWS:
            return not timed and elements > self.TILES_PORTION_ELEMENTS and M <= self.TILES_PORTION_ROWS and \
                work <= self.TILES_PORTION_WORK
        return long or M <= self.TILES_CUT_MAX_ROWS

    LARGE_KINDS = {"plain": 0, "gated": 1, "rotary": 2}

    def _tiled(self, M: int, N: int, K: int, kind: str, tensors, cut_us: Optional[float] = None):
        """((shape, slices), whether in the kernels for many rows) of a product as in `_tiles`, (None, False) if it runs in no
        tiles; `tensors` as in `_large`. One look into what was found before: a step that is launched kernel by kernel comes
        here for every product of every layer."""
        if M < self.LARGE_MIN_ROWS:
            return None, False
        key = (M, N, K, kind, cut_us, self.captured, self.library_timed_rows, self.library_timed_portion)
        try:
            large, tiles = self._large_plans[key]
        except KeyError:
            large, tiles = self._large(M, N, K, kind, (), cut_us), self._tiles(M, N, K, kind, cut_us)
            if len(self._large_plans) >= self.TILE_PLANS:
                self._large_plans.clear()
            self._large_plans[key] = large, tiles
        if large is None:
            return tiles, False
        for t in tensors:
            if t is not None and t.data_ptr() % 16:
                return tiles, False
        return large, True

    def _large(self, M: int, N: int, K: int, kind: str, tensors, cut_us: Optional[float] = None):
        """(shape, slices) of the kernels for many rows for a product as in `_tiles`, None if another kernel is the better one or
        one of the caller's `tensors`, which they take 16 bytes at a time, begins at no multiple of that."""
        if M < self.LARGE_MIN_ROWS or any(t is not None and t.data_ptr() % 16 for t in tensors):
            return None
        shape, slices, us = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_float(0)
        if self._ops.distie_large_tiles_plan(M, N, K, self.LARGE_KINDS[kind], cut_us is not None, cut_us or 0.0,
                                             ctypes.byref(shape), ctypes.byref(slices), ctypes.byref(us)) and \
                self._large_take(M, N, K, kind, cut_us, us.value) and \
                not self._large_idle(M, N, K, kind, cut_us, shape.value, slices.value):
            return shape.value, slices.value
        return None

    def _large_take(self, M, N, K, kind, cut_us, us) -> bool:
        """Whether a product that comes to `us` there, with the reader that adds its slices, is to run so: see the constants."""
        elements = N * K
        if M <= self.LARGE_FEW_ROWS:
            if kind == "gated":
                return M >= (self.LARGE_FEW_GATED_ROWS if elements >= self.LARGE_FEW_GATED_ELEMENTS else self.LARGE_FEW_CUT_ROWS)
            if kind == "plain" and cut_us == 0.0:
                return M >= self.LARGE_FEW_CUT_ROWS and elements >= (self.LARGE_FEW_LONG_ELEMENTS if K >= 2 * N else
                                                                     self.LARGE_FEW_SHORT_ELEMENTS)
            return kind == "plain" and M >= self.LARGE_FEW_CUT_ROWS and elements >= self.LARGE_FEW_HEAD_ELEMENTS
        rate = 2e-6 * M * elements / us
        many = M > self.LARGE_ROWS and (M > self.LARGE_MAX_ROWS or (M * elements > self.LARGE_MANY_ROWS_WORK and K < 5 * N))
        if kind == "gated":
            return rate >= self.LARGE_GATED_RATE
        if kind == "rotary":
            return -(-M // 64) * -(-N // 64) > self._compute_units and rate >= self.LARGE_ROTARY_RATE and \
                (K <= self.LARGE_ROTARY_SHORT_K or -(-M // 64) * -(-N // 128) > self._compute_units) and \
                not many and M * elements <= self.LARGE_ROTARY_WORK and \
                (M >= self.LARGE_ROTARY_ROWS or elements <= self.TILES_LARGE_ROTARY)
        if cut_us != 0.0:
            least = self.LARGE_PLAIN_RATE if N < 4 * K else \
                self.LARGE_WIDE_SHORT_RATE if K <= self.LARGE_WIDE_SHORT_K else self.LARGE_WIDE_RATE
            return rate >= least and M * elements <= self.LARGE_DENSE_WORK
        if many:
            return False
        if K >= 2 * N:
            return rate >= (self.LARGE_LONG_RATE if M <= self.TILES_LONG_ROWS else self.LARGE_LONG_RATE_BEYOND)
        return rate >= (self.LARGE_SHORT_RATE if elements > self.ROW_GROUPS_MAX_ELEMENTS or N < self.TILES_FEW_WEIGHT_ROWS else
                        self.LARGE_SHORT_RATE_SMALL)

    def _large_idle(self, M, N, K, kind, cut_us, shape, slices) -> bool:
        """Whether these tiles leave half of the compute units or more without one where other kernels do not: see LARGE_IDLE_K."""
        if kind == "rotary" or M <= self.LARGE_FEW_ROWS:
            return False
        rows, columns = ctypes.c_int(0), ctypes.c_int(0)
        _check(self._ops.distie_large_tiles_grid(M, N, shape, ctypes.byref(rows), ctypes.byref(columns)), "large_tiles_grid")
        busy = columns.value * slices
        return rows.value == 1 and (4 * busy <= self._compute_units or (2 * busy <= self._compute_units and K > self.LARGE_IDLE_K)) and \
            (M > self._packed_rows(M, N, K) or self._tiles(M, N, K, kind, cut_us) is not None)

    def _large_each(self, M, N, K, xs):
        """The tile of the kernels for many rows for several products that share a launch, N columns in all, or None."""
        if M * N * K > self.LARGE_EACH_WORK or not xs.is_contiguous() or xs.data_ptr() % 16:
            return None
        key = (M, N, K)
        try:
            return self._large_plans[key]
        except KeyError:
            pass
        shape, slices, us = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_float(0)
        plan = None
        if self._ops.distie_large_tiles_plan(M, N, K, 0, 0, 0.0, ctypes.byref(shape), ctypes.byref(slices), ctypes.byref(us)):
            plan = shape.value
        if len(self._large_plans) >= self.TILE_PLANS:
            self._large_plans.clear()
        self._large_plans[key] = plan
        return plan

    def _run_tiles(self, plan, x, packed, bias, out_dtype, M, N, K, gated=0, clamp=(0.0, 1.0, 0.0), large=False):
        """The tiled product; float32 slices if the plan cuts K."""
        shape, slices = plan
        columns = N // 2 if gated else N
        out = self._empty((M, columns), out_dtype) if slices == 1 else \
            self._empty((slices, M, columns), torch.float32)
        kernel, name = (self._ops.distie_large_tiles_bf16, "large_tiles_bf16") if large else \
            (self._ops.distie_packed_tiles_bf16, "packed_tiles_bf16")
        _check(kernel(
            x, packed, bias, out, _code(out),
            M, N, K, gated, shape, slices, *clamp, self._stream()), name)
        return out if slices == 1 else PartialSums(out, out_dtype)

    def _library(self):
        """The vendor library's products, called directly; loaded at the first large product."""
        if self._lib is None:
            lib = ctypes.CDLL(str(build.ensure("library")))
            lib.distie_lib_init.argtypes = [ctypes.c_int]
            lib.distie_lib_init.restype = ctypes.c_int
            lib.distie_lib_linear.argtypes = [_P, _P, _P, _P, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                              ctypes.c_int, ctypes.c_int64, ctypes.c_int, _P]
            lib.distie_lib_linear.restype = ctypes.c_int
            lib.distie_lib_counts.argtypes = [ctypes.POINTER(ctypes.c_long), ctypes.POINTER(ctypes.c_long)]
            lib.distie_lib_counts.restype = None
            lib.distie_lib_more_counts.argtypes = [ctypes.POINTER(ctypes.c_long)] * 3
            lib.distie_lib_more_counts.restype = None
            with torch.cuda.device(self.device):
                _check(lib.distie_lib_init(self._device_index), "lib_init")
            calls.quicken(lib)
            self._lib = lib
        return self._lib

    def library_plans(self):
        """(shapes the library has a plan for, shapes whose kernel was chosen by timing)"""
        made, timed = ctypes.c_long(0), ctypes.c_long(0)
        self._library().distie_lib_counts(ctypes.byref(made), ctypes.byref(timed))
        return made.value, timed.value

    def library_counts(self) -> dict:
        """`held`: shapes the library holds a plan for now; `asked`: how often it was asked to rank its kernels
        (row counts of one class of 32 share a choice); `refused`: timed candidates dropped because their
        result differed from that of the library's first choice."""
        held, asked, refused = ctypes.c_long(0), ctypes.c_long(0), ctypes.c_long(0)
        self._library().distie_lib_more_counts(ctypes.byref(held), ctypes.byref(asked), ctypes.byref(refused))
        return {"held": held.value, "asked": asked.value, "refused": refused.value}

    LIBRARY_UNSUPPORTED = -3

    def _library_linear(self, x, weight, bias, out_dtype):
        """x [M, K] . weight [N, K]^T (+ float32 bias) by the library, float32 sums, into a new [M, N] of `out_dtype`.
        x and weight are both bfloat16, or both float32 (then every product is a float32 product). None if the
        library has no kernel for the product as asked."""
        M, K = x.shape
        N = weight.shape[0]
        if x.stride(1) != 1 or x.stride(0) != K:
            x = x.contiguous()
        if weight.stride(1) != 1 or weight.stride(0) != K:
            weight = weight.contiguous()
        out = self._empty((M, N), out_dtype)
        lib = self._library()
        code, size, w_size = _CODES[out_dtype], out.element_size(), weight.element_size()
        # The library's large bfloat16 kernels work on tiles of 256 x 256, one a compute unit at a time: a product
        # with a few tiles more than a whole number of rounds pays a full round for them (at 2,048 rows 16,384
        # columns take 82 us and 17,920 take 116). The last columns as a product of their own cost less (20 us
        # for 1,536), written into the same output.
        tail = self._library_tail(M, N) if out_dtype == torch.bfloat16 else 0
        for lo, hi in (((0, N - tail), (N - tail, N)) if tail else ((0, N),)):
            rc = lib.distie_lib_linear(
                x.data_ptr(), weight.data_ptr() + lo * K * w_size, bias.data_ptr() + lo * 4 if bias is not None else None,
                out.data_ptr() + lo * size, _code(x), code, M, hi - lo, K, N, 1 if self._tuning else 0, self._stream())
            if rc == self.LIBRARY_UNSUPPORTED:
                return None
            _check(rc, "lib_linear")
        return out

    LIBRARY_TILE = 256

    def _library_tail(self, M: int, N: int) -> int:
        """How many of the last columns of a large library product to run as a product of their own: those
        beyond the last whole round of tiles over the compute units, if they are few (at most a quarter of a
        round) and there is at least one whole round before them; else 0."""
        tile = self.LIBRARY_TILE
        row_tiles = -(-M // tile)
        if row_tiles > self._compute_units:
            return 0
        round_columns = self._compute_units // row_tiles * tile
        tail = N % round_columns
        if N < round_columns or tail == 0 or tail > round_columns // 4 or tail % 8:
            return 0
        return tail

    def _pass_blocks(self, rows: int, elements: int) -> int:
        """Blocks of 16 rows of x per pass of the wide product over a weight of `elements` (0: one pass)."""
        if elements > self.TWO_PASS_MAX_ELEMENTS:
            if rows <= 64:
                return 0
            blocks = -(-rows // 16)
            passes = -(-blocks // self.WIDE_PASS_MAX_BLOCKS)
            return -(-blocks // passes)
        # (a single pass takes at most 64 rows; beyond 128 rows passes of 48 were 5 % faster than of 32 or 64)
        return 0 if rows <= 32 else (2 if rows <= 128 else 3)

    def _rope_table(self, meta, inv_freq):
        """Cosines and sines of the step's positions, float32 [T, pairs, 2]: computed by the first layer
        that asks, used by all."""
        pairs = inv_freq.shape[0]
        key = ("rope", inv_freq.data_ptr(), pairs)
        table = meta.scratch.get(key)
        if table is None:
            table = self._empty((meta.num_tokens, pairs, 2), torch.float32)
            _check(self._ops.distie_rope_table(meta.positions, inv_freq, table,
                                               meta.num_tokens, pairs, self._stream()), "rope_table")
            meta.scratch[key] = table
        return table

    def _linear(self, x, weight, bias, out_dtype, partial_ok=False, lazy=False):
        packed = getattr(weight, "_distie_packed", None)
        if isinstance(x, PendingNorm) and out_dtype == torch.float32 and bias is None and packed is not None and \
                weight.shape[1] == x.shape[1] and weight.dtype == torch.bfloat16:
            # the head behind the final norm
            N, K = weight.shape
            if packed.numel() != self._packed_elements(N, K, False):
                raise KernelError("linear: the packed copy does not belong to this weight")
            out = self._empty((x.shape[0], N), torch.float32)
            return self._norm_product(x, packed, None, out, 0, N)
        x = self.dense(x)
        self._own(x, weight, bias)
        M, K = x.shape
        N = weight.shape[0]
        if weight.shape[1] != K:
            raise KernelError(f"linear: x is [{M}, {K}], weight is {list(weight.shape)}")
        if bias is not None and (bias.dtype != torch.float32 or bias.shape[0] != N):
            raise KernelError("linear: bias must be float32 [N]")
        both_bf16 = x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16
        packed = packed if both_bf16 else None
        if lazy and packed is not None and self._fused(M) and K % 8 == 0 and out_dtype == torch.bfloat16:
            return PendingProduct(x, weight, bias)
        plan, large = None, False
        if packed is not None and weight._distie_role is not None:
            adds = partial_ok and weight._distie_role in self.ADDS_SLICES
            plan, large = self._tiled(M, N, K, "plain", (x, bias), 0.0 if adds else self.SUM_SLICES_US)
        if plan is not None:
            if packed.numel() != self._packed_elements(N, K, False):
                raise KernelError("linear: the packed copy does not belong to this weight")
            out = self._run_tiles(plan, x, packed, bias, out_dtype, M, N, K, large=large)
            return out if partial_ok else self.dense(out)
        if packed is not None and self.ONE_WAVE_MAX_ROWS < M <= self._packed_rows(M, N, K) and K % 8 == 0 and \
                N * K > self.ROW_GROUPS_MAX_ELEMENTS:
            if packed.numel() != self._packed_elements(N, K, False):
                raise KernelError("linear: the packed copy does not belong to this weight")
            slices = self._ops.distie_gemm_packed_wide_slices(N, K)
            if slices == 1:
                out = self._empty((M, N), out_dtype)
            else:
                out = self._empty((slices, M, N), torch.float32)
            _check(self._ops.distie_gemm_packed_wide_bf16(
                x, packed, bias, out,
                _code(out), M, N, K, 0, self._pass_blocks(M, N * K), 0.0, 1.0, 0.0, self._stream()),
                "gemm_packed_wide_bf16")
            if slices == 1:
                return out
            return PartialSums(out, out_dtype) if partial_ok else self.dense(PartialSums(out, out_dtype))
        if both_bf16 and K % 8 == 0 and (M <= self.SKINNY_MAX_ROWS or (packed is not None and M <= self._packed_rows(M, N, K))):
            if packed is not None:
                if packed.numel() != self._packed_elements(N, K, False):
                    raise KernelError("linear: the packed copy does not belong to this weight")
            slices = self._ops.distie_gemm_skinny_slices(M, N, K)       # the same cut for both kernels
            if slices == 1:
                out = self._empty((M, N), out_dtype)
            else:
                out = self._empty((slices, M, N), torch.float32)
            if packed is not None:
                _check(self._ops.distie_gemm_packed_bf16(
                    x, packed, bias, out,
                    _code(out), M, N, K, 0, 0.0, 1.0, 0.0, self._stream()), "gemm_packed_bf16")
            else:
                _check(self._ops.distie_gemm_skinny_bf16(
                    x, weight, bias, out,
                    _code(out), M, N, K, self._stream()), "gemm_skinny_bf16")
            if slices == 1:
                return out
            return PartialSums(out, out_dtype) if partial_ok else self.dense(PartialSums(out, out_dtype))
        if both_bf16:
            # large bfloat16 product: the library's matrix-core kernels
            out = self._library_linear(x, weight, bias, out_dtype)
            if out is None:
                # no kernel of the library's for this product as asked for: through torch, which knows more ways
                out = torch.mm(x, weight.t(), out_dtype=torch.float32)
                out = out if bias is None else out + bias
                out = out if out_dtype == torch.float32 else out.to(out_dtype)
            return out
        both_f32 = x.dtype == torch.float32 and weight.dtype == torch.float32 and out_dtype == torch.float32
        if both_f32 and M > self.ROWS_MAX_ROWS:
            # large float32 product: the library's float32 kernels (float32 products and sums); else the generic one
            out = self._library_linear(x, weight, bias, out_dtype)
            if out is not None:
                return out
        if both_f32 and partial_ok:
            # few rows in the true 32-bit path, for a caller that takes slices (the head's product does not, and runs at 5
            # TB/s as it is): the weights streamed through the matrix cores' float32 products
            slices = self._ops.distie_rows_f32_slices(M, N, K, 0) if self._rows_f32_take(M, N, K) else 0
            if slices:
                out = self._empty((M, N) if slices == 1 else (slices, M, N), torch.float32)
                _check(self._ops.distie_rows_f32(
                    x, weight, bias, out, M, N, K,
                    0, slices, 0.0, 1.0, 0.0, self._stream()), "rows_f32")
                return out if slices == 1 else PartialSums(out, out_dtype)
        out = self._empty((M, N), out_dtype)
        if M <= self.ROWS_MAX_ROWS and K % 8 == 0:
            # few rows in float32 (or against a weight kept in float32): the weights are streamed, FMAs only
            _check(self._ops.distie_gemv_rows(
                x, _code(x), weight, _code(weight), bias,
                out, _CODES[out_dtype], M, N, K, self._stream()), "gemv_rows")
            return out
        _check(self._ops.distie_gemm_generic(
            x, _code(x), weight, _code(weight), bias,
            out, _CODES[out_dtype], M, N, K, self._stream()), "gemm_generic")
        return out

    def _rows_f32_take(self, M, N, K) -> bool:
        """Whether a plain float32 product of few rows is the faster one on the matrix cores: see the constants."""
        if N * K < self.ROWS_F32_MIN_ELEMENTS:
            return False
        if M <= 4:
            return N * K >= self.ROWS_F32_FEW_ELEMENTS and (K >= 4 * N and N <= 4096 if M == 1 else K >= 2 * N)
        if M <= 8:
            return N * K > self.ROWS_F32_EIGHT_ELEMENTS
        return N >= (768 if 16 < M <= 24 else 640)

    def linear(self, x, weight, bias=None):
        """May return `PartialSums` (see there)."""
        return self._linear(x, weight, bias, x.dtype, partial_ok=True, lazy=True)

    def linear_dense(self, x, weight, bias=None):
        """Steps of up to ONE_WAVE_MAX_ROWS rows: the packed product with the whole K in one workgroup, which writes the
        finished values (cut into slices, a kernel that adds them up would have to follow)."""
        x = self.dense(x)
        packed = getattr(weight, "_distie_packed", None)
        M, K = x.shape
        N = weight.shape[0]
        if packed is None or x.dtype != torch.bfloat16 or M > self.ONE_WAVE_MAX_ROWS or K % 8 or weight.shape[1] != K:
            return self.dense(self.linear(x, weight, bias))
        self._own(x, bias)
        if bias is not None and (bias.dtype != torch.float32 or bias.shape[0] != N):
            raise KernelError("linear: bias must be float32 [N]")
        if packed.numel() != self._packed_elements(N, K, False):
            raise KernelError("linear: the packed copy does not belong to this weight")
        out = self._empty((M, N), x.dtype)
        _check(self._ops.distie_gemm_packed_bf16(
            x, packed, bias, out, _code(out), M, N, K,
            2, 0.0, 1.0, 0.0, self._stream()), "gemm_packed_bf16")
        return out

    def linear_f32out(self, x, weight, bias=None, scale=1.0, partial=False):
        if partial and scale == 1.0:
            return self._linear(x, weight, bias, torch.float32, partial_ok=True)
        out = self._linear(x, weight, bias, torch.float32)
        if scale != 1.0:
            _check(self._ops.distie_scale_f32(out, out.numel(), float(scale), self._stream()), "scale_f32")
        return out

    def rope_kv_write(self, qkv, meta: BatchMeta, group, k_cache, v_cache, inv_freq, num_heads, num_kv_heads,
                      head_dim, write):
        if isinstance(qkv, (PendingNorm, PendingProduct)):
            qkv = self.dense(qkv)
        slices, source = 1, qkv
        if isinstance(qkv, PartialSums):
            slices, source = qkv.slices, qkv.data
            out = self._empty(tuple(qkv.shape), qkv.dtype)
        else:
            out = qkv
        self._own(source, k_cache, v_cache, inv_freq)
        T = out.shape[0]
        if out.shape[1] != (num_heads + 2 * num_kv_heads) * head_dim:
            raise KernelError("rope_kv_write: qkv width does not match the head counts")
        self._check_cache(k_cache, v_cache, num_kv_heads, meta.block_size, head_dim)
        if T != meta.num_tokens:
            raise KernelError("rope_kv_write: qkv rows do not match the batch")
        pairs = 0 if inv_freq is None else inv_freq.shape[0]
        slots = meta.groups[group].slots
        table = self._rope_table(meta, inv_freq) if pairs else None
        _check(self._ops.distie_rope_kv_write(
            source, _code(source), slices, out, _code(out),
            table, meta.positions,
            slots, k_cache, v_cache, _code(k_cache),
            inv_freq, pairs, T, num_heads, num_kv_heads, head_dim,
            meta.block_size, 1 if write else 0, self._stream()), "rope_kv_write")
        _mark_written(out)
        return out

    def paged_attention(self, qkv, meta: BatchMeta, group, k_cache, v_cache, num_heads, num_kv_heads, head_dim,
                        scale, window, extras=None):
        """The matrix-core kernels and the tiled float32 kernel compute attention with plain scores (a sink in the
        denominator they take, and chunks instead of a window); a step whose `extras` bend the scores goes to the
        wave-per-token kernel, which takes slopes and a cap as well (any types and sizes)."""
        if not scale > 0:
            raise KernelError(f"paged_attention: the scale of the scores must be positive, not {scale}")
        qkv = self.dense(qkv)
        self._own(qkv, k_cache, v_cache)
        T = qkv.shape[0]
        table = meta.groups[group].block_table
        self._check_cache(k_cache, v_cache, num_kv_heads, meta.block_size, head_dim)
        rows = meta.table_rows
        if T != meta.num_tokens or (rows is None and table.shape[0] != meta.num_requests) or \
                (rows is not None and rows.shape[0] != meta.num_requests):
            raise KernelError("paged_attention: tensors do not match the batch")
        rows_ptr = rows
        out = self._empty((T, num_heads * head_dim), qkv.dtype)
        plain = extras is None or not extras.bends_scores
        slopes, cap = (None, 0.0) if plain else (extras.head_slopes, float(extras.score_cap or 0.0))
        sinks = extras.sinks if extras is not None else None
        for name, vector in (("head_slopes", slopes), ("sinks", sinks)):
            if vector is not None:
                self._own(vector)
                if vector.dtype != torch.float32 or tuple(vector.shape) != (num_heads,):
                    raise KernelError(f"paged_attention: {name} must be float32 [num_heads]")
        sinks_ptr = sinks
        chunk = extras.chunk if extras is not None else 0
        if chunk and (window or extras.mixes_heads):
            raise KernelError("paged_attention: chunks do not go with a window or with mixed heads")
        reach = -int(chunk) if chunk else int(window or 0)       # as the kernels take it: a window, or minus the chunks' size
        if extras is not None and extras.mixes_heads:
            self._mixed_attention(qkv, meta, table, rows_ptr, k_cache, v_cache, out, num_heads, num_kv_heads, head_dim, scale,
                                  window, extras)
            return out
        lib = self.attention_library(head_dim)
        bf16 = qkv.dtype == torch.bfloat16 and k_cache.dtype == torch.bfloat16
        if plain and bf16 and meta.block_size % 16 == 0 and head_dim % 16 == 0 and head_dim <= self.LARGEST_MATRIX_CORE_HEAD:
            # how the step is launched, and its buffers for partial results, are the same for every layer
            # with these sizes: worked out once per step (the layers run one after the other, so they can
            # share the buffers)
            key = ("attention", reach, num_heads, num_kv_heads, head_dim, meta.max_kv, meta.all_decode,
                   meta.singles_bound, *(getattr(self, name) for name in self.ATTENTION_PLAN_RULES))
            plan = meta.scratch.get(key)
            if plan is None or plan["cu_q"] is not meta.host_cu_q:
                plan = meta.scratch[key] = self._attention_plan(lib, meta, T, num_heads, num_kv_heads, head_dim, abs(reach))
            if plan["decode"]:
                _check(lib.distie_attention_decode_bf16(
                    qkv, qkv.shape[1], k_cache, v_cache, meta.kv_len,
                    meta.cu_q, table, table.shape[1], rows_ptr, out,
                    plan["decode_o"], plan["decode_ml"], meta.num_requests, num_heads,
                    num_kv_heads, meta.block_size, float(scale), reach, plan["split_len"],
                    plan["max_splits"], 1 if meta.all_decode else 0,
                    plan["run_len"], sinks_ptr, plan["together"],
                    self._stream()), "attention_decode_bf16")
            if plan["prefill"] and plan["waves"]:
                _check(lib.distie_attention_prefill_keys(
                    qkv, qkv.shape[1], k_cache, v_cache, meta.positions,
                    meta.cu_q, table, table.shape[1], rows_ptr, out, T, meta.num_requests,
                    num_heads, num_kv_heads, meta.block_size, float(scale), reach, 2 if plan["decode"] else 1, sinks_ptr,
                    plan["waves"], self._stream()), "attention_prefill_keys")
            elif plan["prefill"]:
                parts = plan["parts"]
                _check(lib.distie_attention_prefill_bf16(
                    qkv, qkv.shape[1], k_cache, v_cache, meta.positions,
                    meta.cu_q, table, table.shape[1], rows_ptr, out, T, meta.num_requests,
                    num_heads, num_kv_heads, meta.block_size, float(scale), reach,
                    2 if plan["decode"] else 1, meta.token_request,
                    plan["prefill_o"] if parts > 1 else None,
                    plan["prefill_ml"] if parts > 1 else None, parts, sinks_ptr, self._stream()),
                    "attention_prefill_bf16")
            return out
        f32 = qkv.dtype == torch.float32 and k_cache.dtype == torch.float32
        if plain and f32 and meta.max_q >= self.PREFILL_F32_MIN_TOKENS and meta.block_size % 16 == 0 and \
                qkv.shape[1] % 4 == 0 and lib.distie_attention_prefill_f32_fits():
            # portions of prompts in float32: the tiled kernel on float32 matrix products takes the whole step
            key = ("attention_f32", reach, num_heads, head_dim, meta.max_kv, self.PREFILL_PARTS,
                   self.PREFILL_WORKGROUPS)
            plan = meta.scratch.get(key)
            if plan is None:
                plan = meta.scratch[key] = self._prefill_parts(meta, T, meta.max_kv, num_heads, head_dim, abs(reach))
            parts = plan["parts"]
            _check(lib.distie_attention_prefill_f32(
                qkv, qkv.shape[1], k_cache, v_cache, meta.positions,
                meta.cu_q, table, table.shape[1], rows_ptr, out, T, meta.num_requests,
                num_heads, num_kv_heads, meta.block_size, float(scale), reach, 1,
                meta.token_request, plan["prefill_o"] if parts > 1 else None,
                plan["prefill_ml"] if parts > 1 else None, parts, sinks_ptr, self._stream()),
                "attention_prefill_f32")
            return out
        columns, runs, per, waves = 0, 1, 0, 0
        if plain and f32:
            # which kernel takes the step and how it is cut: the same for every layer with these sizes
            aligned = (qkv.data_ptr() | k_cache.data_ptr() | v_cache.data_ptr()) % 16 == 0
            key = ("attention_f32_plan", reach, num_heads, num_kv_heads, head_dim, qkv.shape[1], meta.max_kv, aligned)
            plan = meta.scratch.get(key)
            if plan is None:
                plan = meta.scratch[key] = self._plan_f32(lib, meta, T, num_heads, num_kv_heads, qkv.shape[1], abs(reach), aligned)
            columns, runs, per, waves = plan
        part_o, part_ml = self._run_parts(meta, runs, T, num_heads, head_dim)
        if columns:
            # wide heads, or many tokens: a tile of tokens and a kv head's query heads are the columns of matrix products
            _check(lib.distie_attention_columns_f32(
                qkv, qkv.shape[1], k_cache, v_cache, meta.positions,
                meta.cu_q, table, table.shape[1], rows_ptr, out, T, meta.num_requests,
                num_heads, num_kv_heads, meta.block_size, float(scale), reach, sinks_ptr,
                part_o if runs > 1 else None, part_ml if runs > 1 else None, runs, self._stream()),
                "attention_columns_f32")
            return out
        _check(lib.distie_attention_generic(
            qkv, _code(qkv), qkv.shape[1], k_cache, v_cache, _code(k_cache),
            meta.positions, meta.token_request, table, table.shape[1], rows_ptr,
            out, T, num_heads, num_kv_heads, meta.block_size, float(scale), reach,
            slopes, cap, sinks_ptr, part_o if runs > 1 else None,
            part_ml if runs > 1 else None, runs, per, waves, self._stream()), "attention_generic")
        return out

    def _mixed_attention(self, q, meta: BatchMeta, table, rows_ptr, k_cache, v_cache, out, num_heads, num_kv_heads, head_dim,
                         scale, window, extras) -> None:
        """Attention for layers whose heads see each other's scores (csrc/mixed_attention.hip)."""
        if extras.head_slopes is not None:
            raise KernelError("paged_attention: slopes do not go with mixed heads")
        bias, mix = extras.distance_bias, extras.head_mix
        for name, t, rows in (("distance_bias", bias, num_heads), ("head_mix", mix, num_heads)):
            if t is not None:
                self._own(t)
                if t.dtype != torch.float32 or t.dim() != 2 or t.shape[0] != rows:
                    raise KernelError(f"paged_attention: {name} must be float32 with a row a head")
        if mix is not None and mix.shape[1] != num_heads:
            raise KernelError("paged_attention: head_mix must be [num_heads, num_heads]")
        if q.shape[1] != num_heads * head_dim:
            raise KernelError("paged_attention: mixed heads take q alone")
        keep = int(extras.keep_first) if window else 0
        if q.dtype == torch.bfloat16 and k_cache.dtype == torch.bfloat16 and meta.block_size % 16 == 0 and \
                head_dim % 32 == 0 and head_dim <= self.LARGEST_MATRIX_CORE_HEAD:
            lib = self.mixed_attention_library(head_dim)
            queries = lib.distie_mixed_fits(num_heads, num_kv_heads)
            if queries:
                key = ("mixed_attention", int(window or 0), keep, num_heads, head_dim, meta.max_kv, meta.all_decode,
                       meta.singles_bound)
                plan = meta.scratch.get(key)
                if plan is None or plan["cu_q"] is not meta.host_cu_q:
                    plan = meta.scratch[key] = self._mixed_plan(lib, meta, num_heads, head_dim, window, keep)
                if queries == 16 and q.shape[0] < self.MIXED_WIDE_TOKENS:
                    queries = 8
                _check(lib.distie_mixed_attention_bf16(
                    q, q.shape[1], k_cache, v_cache, meta.positions,
                    meta.cu_q, table, table.shape[1], rows_ptr, out, q.shape[0],
                    meta.num_requests, num_heads, num_kv_heads, meta.block_size, float(scale), int(window or 0), keep,
                    float(extras.score_cap or 0.0), bias, bias.shape[1] if bias is not None else 0, mix,
                    extras.sinks, 1 if plan["prefill"] else 0, queries, (2 if meta.all_decode else 1) if plan["decode"] else 0, plan["splits"],
                    plan["partial_o"], plan["partial_ml"], self._stream()), "mixed_attention_bf16")
                return
        if not self._ops.distie_mixed_attention_fits(num_heads, head_dim):
            raise KernelError(f"paged_attention: {num_heads} mixed heads of {head_dim} do not fit the LDS of a compute unit")
        _check(self._ops.distie_mixed_attention_generic(
            q, _code(q), q.shape[1], k_cache, v_cache, _code(k_cache),
            meta.positions, meta.token_request, table, table.shape[1], rows_ptr,
            out, q.shape[0], num_heads, num_kv_heads, head_dim, meta.block_size, float(scale), int(window or 0),
            keep, float(extras.score_cap or 0.0), bias, bias.shape[1] if bias is not None else 0, mix,
            extras.sinks, self._stream()), "mixed_attention_generic")

    def _mixed_plan(self, lib, meta: BatchMeta, num_heads, head_dim, window, keep) -> dict:
        """Which of the mixed heads' kernels a step needs, and the buffers for partial results of single tokens (one
        for every run of keys a token may see): the same for every layer with these sizes."""
        singles = meta.num_requests if meta.all_decode else 0
        if not meta.all_decode and meta.singles_bound is not None:
            singles = meta.singles_bound
        elif not meta.all_decode and meta.host_cu_q is not None:
            singles = int((meta.host_cu_q[1:] - meta.host_cu_q[:-1] == 1).sum())
        run = lib.distie_mixed_decode_keys()
        plan = {"cu_q": meta.host_cu_q, "decode": singles > 0, "splits": 0, "partial_o": None, "partial_ml": None,
                "prefill": singles < meta.num_requests or (meta.singles_bound is not None and not meta.all_decode)}
        if plan["decode"]:
            splits = -(-meta.max_kv // run)
            if window:
                splits = min(splits, -(-keep // run) + (int(window) + run - 2) // run + 1)
            plan["splits"] = max(1, splits)
            shape = (meta.num_requests, plan["splits"], num_heads)
            plan["partial_o"] = self._empty((*shape, head_dim), torch.float32)
            plan["partial_ml"] = self._empty((*shape, 2), torch.float32)
        return plan

    COLUMNS_KEYS = 32                # a window's keys begin anywhere in a chunk of so many

    @classmethod
    def _columns_runs(cls, lib, T, requests, num_heads, num_kv_heads, block_size, stride, max_kv, reach):
        """The runs of the float32 kernel in columns, 0 where it does not take the step or another kernel is faster."""
        runs = lib.distie_attention_columns_f32_runs(T, requests, num_heads, num_kv_heads, block_size, stride,
                                                     min(max_kv, reach or max_kv))
        if runs > 0:
            spans = min(max_kv, reach + cls.COLUMNS_KEYS - 1) if reach else max_kv
            if not lib.distie_attention_columns_f32_pays(T, requests, num_heads, num_kv_heads, block_size, spans, runs):
                return 0
        return runs

    def _plan_f32(self, lib, meta: BatchMeta, T, num_heads, num_kv_heads, stride, reach, aligned):
        """(in columns, runs of keys, heads a workgroup, waves) of a float32 step with plain scores. The keys of a token can be
        cut into runs that run side by side, so that few requests occupy the chip as well."""
        runs = self._columns_runs(lib, T, meta.num_requests, num_heads, num_kv_heads, meta.block_size, stride, meta.max_kv,
                                  reach) if aligned else 0
        if runs > 0:
            return True, runs, 0, 0
        return (False, *self._grouped_plan(lib, T, num_heads, num_kv_heads, min(meta.max_kv, reach or meta.max_kv)))

    @staticmethod
    def _grouped_plan(lib, T, num_heads, num_kv_heads, visible):
        """(runs, heads a workgroup, waves) of the float32 kernel for few pairs of token and head."""
        per, waves = ctypes.c_int(0), ctypes.c_int(0)
        runs = lib.distie_attention_f32_plan(T, num_heads, num_kv_heads, visible, ctypes.byref(per), ctypes.byref(waves))
        return runs, per.value, waves.value

    def _run_parts(self, meta: BatchMeta, runs, T, num_heads, head_dim):
        """The buffers for the sums of `runs` runs of keys, kept for the step's layers."""
        if runs == 1:
            return None, None
        key = ("attention_f32_runs", runs, num_heads, head_dim)
        held = meta.scratch.get(key)
        if held is None:
            held = meta.scratch[key] = (
                self._empty((runs, T, num_heads, head_dim), torch.float32),
                self._empty((runs, T, num_heads, 2), torch.float32))
        return held

    def _attention_plan(self, lib, meta: BatchMeta, T, num_heads, num_kv_heads, head_dim, window) -> dict:
        group = num_heads // num_kv_heads
        singles = meta.num_requests if meta.all_decode else 0
        if not meta.all_decode and meta.singles_bound is not None:
            # a captured step of portions and single tokens: which requests bring one token is known on the device
            # only; both kernels are launched for as many as there may be, and each leaves the other's requests alone
            singles = meta.singles_bound
        elif not meta.all_decode and meta.host_cu_q is not None:
            singles = int((meta.host_cu_q[1:] - meta.host_cu_q[:-1] == 1).sum())
        plan = {"cu_q": meta.host_cu_q, "decode": singles > 0 and group <= lib.distie_attention_decode_columns()}
        if plan["decode"]:
            # requests that bring one token: keys are cut into runs, one wave each, so that the chip is
            # filled even when few requests decode. The kernel cuts every request's visible keys (counted
            # from a 64-key boundary) into at most `max_splits` runs by the request's own length; the length
            # of the longest request's runs is passed along as a hint for the first lookups of pages.
            visible = min(meta.max_kv, int(window) + 63) if window else meta.max_kv
            max_splits = max(1, min(self.DECODE_MAX_RUNS, self.DECODE_WAVES // (singles * num_kv_heads),
                                    -(-visible // 64)))
            plan["split_len"] = -(-visible // (64 * max_splits)) * 64
            # every request with one token, no window, waves left over: one run length for all of them, so that a
            # long request gets more runs than a short one (up to twice what every request would get)
            plan["run_len"] = None
            pairs = singles * num_kv_heads
            if meta.all_decode and not window and max_splits * pairs <= self.DECODE_SHARED_BELOW * self.DECODE_WAVES:
                splits = max_splits
                max_splits = max(1, min(self.DECODE_MAX_RUNS, 2 * splits, -(-visible // 64)))
                plan["run_len"] = self._empty(1, torch.int32)
                _check(lib.distie_attention_decode_run_len(meta.kv_len, meta.num_requests,
                                                           max(1, self.DECODE_WAVES // num_kv_heads), max_splits,
                                                           plan["run_len"], self._stream()),
                       "attention_decode_run_len")
            plan["max_splits"] = max_splits
            # many runs: a workgroup puts consecutive ones together before it writes their result
            plan["together"] = together = lib.distie_attention_decode_together(max_splits, group, pairs)
            places = -(-max_splits // together)
            plan["decode_o"] = self._empty((meta.num_requests, num_heads, places, head_dim), torch.float32)
            plan["decode_ml"] = self._empty((meta.num_requests, num_heads, places, 2), torch.float32)
        plan["prefill"] = singles < meta.num_requests or not plan["decode"] or \
            (meta.singles_bound is not None and not meta.all_decode)
        if plan["prefill"]:
            keys = self._portions_keys(meta) if plan["decode"] else meta.max_kv
            plan["waves"] = self._prefill_waves(lib, meta, T, singles if plan["decode"] else 0, keys, num_heads, num_kv_heads, window)
            if not plan["waves"]:
                plan.update(self._prefill_parts(meta, T, keys, num_heads, head_dim, window))
        return plan

    @staticmethod
    def _portions_keys(meta: BatchMeta) -> int:
        """The most keys that a request with more than one token has: what a request decodes behind is nothing to the portions
        beside it. Where the host does not know the requests (captured steps) the longest that any may have. By the longest context
        of all before, us of both kernels: 12 heads, 300 tokens beside one request of 5,000 keys 30.7 -> 18.2, beside 24 of 900 22.0 ->
        19.5; 28 heads, 3 prompts of 667 beside one of 5,000 66 -> 39, beside 4 of 16,000 114 -> 56, beside 24 of 1,500 (two waves ->
        tiled) 51 -> 53 with the prompts in front, 55 either way behind the others, where the engine puts them."""
        if meta.host_cu_q is None or meta.host_past is None:
            return meta.max_kv
        tokens = np.diff(np.asarray(meta.host_cu_q))
        return int((np.asarray(meta.host_past) + tokens)[tokens > 1].max(initial=1))

    def _prefill_waves(self, lib, meta: BatchMeta, T, singles, keys, num_heads, num_kv_heads, window) -> int:
        """How many waves of a workgroup share a tile of 32 tokens of the portions of prompts and split its keys; 0: the tiled
        kernel, whose waves share the keys."""
        if not self.PREFILL_PARTS or not lib.distie_attention_prefill_keys_fits(num_kv_heads, meta.block_size) or \
                -(-T // 32) + meta.num_requests > 65535:
            return 0
        visible = min(keys, int(window) + 32) if window else keys
        tokens, portions = max(1, T - singles), max(1, meta.num_requests - singles)
        workgroups = num_heads * (-(-tokens // 32) + portions // 2)
        many, far, times = self.PREFILL_WAVES_BEHIND
        reach = next(reach for most, reach in self.PREFILL_WAVES_REACH if most is None or workgroups <= most)
        if visible > reach * self.PREFILL_PARTS[0][0] or \
                (tokens < self.PREFILL_WAVES_FEW[0] and visible > self.PREFILL_WAVES_FEW[1]) or \
                (workgroups > many and visible > far and visible * portions >= times * tokens) or \
                any(workgroups > least and visible < most for least, most in self.PREFILL_WAVES_MANY):
            return 0
        for waves, most, least in self.PREFILL_WAVES:
            if workgroups <= most and visible >= least:
                return waves
        return 2

    def _prefill_parts(self, meta: BatchMeta, T, keys, num_heads, head_dim, window) -> dict:
        """Into how many parts the tiled kernel cuts its walk over up to `keys` keys, and the buffers between it and the
        merge. Portions of prompts (and single tokens too, if no other kernel took them): long walks over the
        keys are cut into parts that run side by side."""
        visible = min(keys, int(window) + 128) if window else keys
        parts = 1
        for least, cut in self.PREFILL_PARTS:
            if visible >= least:
                parts = cut
        # few new tokens make few workgroups (one per 128 tokens of a request and head), each walking all
        # the keys alone: more parts then, down to 128 keys a part
        tiles = -(-T // 128) + meta.num_requests
        wanted = -(-self.PREFILL_WORKGROUPS // (tiles * num_heads))
        parts = max(parts, min(wanted, visible // 128, 16))
        plan = {"parts": parts}
        if parts > 1:
            plan["prefill_o"] = self._empty((parts, T, num_heads, head_dim), torch.float32)
            plan["prefill_ml"] = self._empty((parts, T, num_heads, 2), torch.float32)
        return plan

    # ---- residual streams, convolutions over time, decayed states, gates (csrc/sequence.hip)
    def _rows_view(self, t: torch.Tensor, width: int):
        """(pointer, row stride) of a [T, width] tensor or column view whose rows are contiguous."""
        if t.device != self.device or t.dim() != 2 or t.shape[1] != width or (t.shape[1] > 1 and t.stride(1) != 1):
            raise KernelError("kernels take row views with contiguous columns on their own device")
        return t.data_ptr(), t.stride(0)

    NORM_KINDS = {"none": 0, "layer": 1, "rms": 2}
    # a step in which some request brings at least so many rows runs the decayed state in chunks of rows that are
    # worked side by side (three kernels) instead of row after row (one)
    SCAN_CHUNKED_MIN_ROWS = 16
    LRU_CHUNKED_MIN_ROWS = 128       # the same for the scan of a channel-wise recurrence (chunks of 64 rows, two kernels)
    ACTIVATIONS = {"relu2": 0, "silu": 1, "gelu_tanh": 2, "relu": 3}

    def hyper_step(self, streams, *, init=None, delta=None, gate=None, mix=None, write=None, read=None,
                   norm_weight=None, norm="none", eps=0.0, out_dtype=None):
        if norm not in self.NORM_KINDS:
            raise KernelError(f"no norm named {norm!r}")
        if init is not None:
            if streams is not None or mix is None and write is None and read is None:
                raise KernelError("hyper_step: `init` makes the streams; it needs their number from mix, write or read")
            self._own(init)
            count = (read if read is not None else write).shape[0]
            if init.dtype != torch.float32 or init.dim() != 2:
                raise KernelError("hyper_step: init must be float32 [T, C]")
            streams = self._empty((init.shape[0], count, init.shape[1]), torch.float32)
        self._own(streams, mix, write, read, norm_weight)
        if streams.dtype != torch.float32 or streams.dim() != 3:
            raise KernelError("hyper_step: streams must be float32 [T, S, C]")
        T, S, C = streams.shape
        for name, t, shape in (("mix", mix, (S, S)), ("write", write, (S,)), ("read", read, (S,))):
            if t is not None and (t.dtype != torch.float32 or tuple(t.shape) != shape):
                raise KernelError(f"hyper_step: {name} must be float32 {list(shape)}")
        if init is not None and tuple(init.shape) != (T, C):
            raise KernelError("hyper_step: init does not match the streams")
        slices, y, y_code, g_ptr, g_code, g_ld, g_slices = 1, None, _F32, None, _F32, 0, 1
        if delta is not None:
            if mix is None or write is None:
                raise KernelError("hyper_step: a delta needs mix and write weights")
            if isinstance(delta, (PendingNorm, PendingProduct)):
                delta = self.dense(delta)
            if isinstance(delta, PartialSums):
                slices, delta = delta.slices, delta.data
            self._own(delta)
            if tuple(delta.shape[-2:]) != (T, C):
                raise KernelError("hyper_step: delta must be [T, C]")
            y, y_code = delta.data_ptr(), _code(delta)
            if gate is not None:
                if isinstance(gate, (PendingNorm, PendingProduct)):
                    gate = self.dense(gate)
                if isinstance(gate, PartialSums):
                    g_slices, gate = gate.slices, gate.data
                    self._own(gate)
                    if tuple(gate.shape[-2:]) != (T, C):
                        raise KernelError("hyper_step: the gate must be [T, C]")
                    g_ptr, g_ld = gate.data_ptr(), C
                else:
                    g_ptr, g_ld = self._rows_view(gate, C)
                g_code = _code(gate)
        h = None
        if read is not None:
            if norm != "none" and (norm_weight is None or tuple(norm_weight.shape) != (C,)):
                raise KernelError("hyper_step: the norm needs a weight [C]")
            h = self._empty((T, C), out_dtype or torch.float32)
        _check(self._ops.distie_hyper_step(
            streams, S, init, y, y_code, slices, g_ptr, g_code, g_ld, g_slices, mix, write, read,
            norm_weight, _code(norm_weight) if norm_weight is not None else _F32, self.NORM_KINDS[norm], float(eps),
            h, _code(h) if h is not None else _F32, T, C, self._stream()), "hyper_step")
        _mark_written(streams)
        return streams, h

    def causal_conv(self, x, weight, state, meta, residual=False, bias=None, act=None):
        if act is not None and act not in self.ACTIVATIONS:
            raise KernelError(f"causal_conv: no activation named {act!r}")
        x = self.dense(x)
        self._own(weight, state, bias)
        T, N = x.shape
        x_ptr, ldx = self._rows_view(x, N)
        taps = weight.shape[1]
        if tuple(weight.shape) != (N, taps) or T != meta.num_tokens:
            raise KernelError("causal_conv: weight must be [channels of x, taps], x the step's rows")
        if bias is not None and (bias.dtype != torch.float32 or tuple(bias.shape) != (N,)):
            raise KernelError("causal_conv: bias must be float32 [channels]")
        self._check_conv_state(state, taps, N)
        out = self._empty((T, N), x.dtype)
        _check(self._ops.distie_causal_conv(
            x_ptr, _code(x), ldx, weight, _code(weight), taps, state if taps > 1 else None,
            out, _code(out), N, (1 if residual else 0) | (0 if act is None else (self.ACTIVATIONS[act] + 1) << 1),
            bias,
            meta.cu_q, meta.token_request, meta.state_slots, T, N, self._stream()),
            "causal_conv")
        if taps > 1 and not meta.all_decode:
            # requests that bring one row moved their state on in the kernel above; the others here, once all
            # rows of the step have read the old one
            _check(self._ops.distie_conv_state(x_ptr, _code(x), ldx, taps, state, meta.cu_q,
                                               meta.state_slots, meta.num_requests, N, 1, self._stream()),
                   "conv_state")
        if taps > 1:
            _mark_written(state)
        return out

    def _check_conv_state(self, state, taps, channels) -> None:
        if taps > 1 and (state is None or state.dtype != torch.float32 or tuple(state.shape[1:]) != (taps - 1, channels)):
            raise KernelError(f"the state of a convolution of {taps} taps over {channels} channels is float32 "
                              f"[slots, {taps - 1}, {channels}]")

    def conv_rope_kv_write(self, product, conv_weight, state, meta, group, k_cache, v_cache, inv_freq, magnitude,
                           num_heads, num_kv_heads, dim, value_dim, padded_dim, has_kv, write, q_temp=None, qk_norm=None,
                           keys_are_values=False, neighbours=False):
        # without a filter the kernel adds up a product's partial sums itself while it reads them
        slices, q_dtype = 1, None
        if isinstance(product, PartialSums) and conv_weight is None:
            slices, q_dtype, product = product.slices, product.dtype, product.data.view(-1, product.data.shape[-1])
        else:
            product = self.dense(product)
            q_dtype = product.dtype
        q_norm = k_norm = None
        norm_eps = 0.0
        if qk_norm is not None:
            q_norm, k_norm, norm_eps = qk_norm
            self._own(q_norm, k_norm)
            for weight in (q_norm, k_norm):
                if weight is not None and (weight.dtype != torch.float32 or tuple(weight.shape) != (dim,)):
                    raise KernelError("conv_rope_kv_write: the norms' weights of q and k are float32 [dim]")
            if q_norm is None or (has_kv and k_norm is None):
                raise KernelError("conv_rope_kv_write: a norm on the heads needs a weight for q, and for k where there are keys")
        self._own(product, conv_weight, state, k_cache, v_cache, inv_freq)
        T, W = product.shape[0] // slices, product.shape[1]
        if keys_are_values and (not has_kv or conv_weight is not None or value_dim != dim):
            raise KernelError("conv_rope_kv_write: values that are the keys go with keys, one head size and no filter")
        channels = num_heads * dim + (num_kv_heads * (dim if keys_are_values else dim + value_dim) if has_kv else 0)
        taps = 0 if conv_weight is None else conv_weight.shape[1]
        if T != meta.num_tokens or W < channels:
            raise KernelError("conv_rope_kv_write: the product does not match the batch or the head counts")
        if conv_weight is not None and tuple(conv_weight.shape) != (channels, taps):
            raise KernelError(f"conv_rope_kv_write: the filters must be [{channels}, taps]")
        self._check_conv_state(state, taps, channels)
        write = bool(write and has_kv)
        if write:
            self._check_cache(k_cache, v_cache, num_kv_heads, meta.block_size, padded_dim)
            if k_cache.dtype != v_cache.dtype:
                raise KernelError("conv_rope_kv_write: keys and values are cached in one dtype")
        pairs = 0 if inv_freq is None else inv_freq.shape[0]
        table = self._rope_table(meta, inv_freq) if pairs else None
        q = self._empty((T, num_heads * padded_dim), q_dtype)
        _check(self._ops.distie_conv_rope_kv_write(
            product, _code(product), W, conv_weight, _code(conv_weight) if conv_weight is not None else _F32,
            taps, state if taps > 1 else None, table, pairs, float(magnitude), q,
            k_cache if write else None, v_cache if write else None, _code(k_cache) if write else _code(product),
            meta.groups[group].slots if write else None, meta.cu_q, meta.token_request,
            meta.state_slots, T, num_heads, num_kv_heads, dim, value_dim, padded_dim, meta.block_size,
            2 if keys_are_values else (1 if has_kv else 0), 1 if write else 0, meta.positions, float(q_temp[0]) if q_temp else 0.0,
            int(q_temp[1]) if q_temp else 0, q_norm, k_norm if has_kv else None, float(norm_eps),
            slices, _CODES[q_dtype], 1 if neighbours else 0, self._stream()), "conv_rope_kv_write")
        if taps > 1:
            if not meta.all_decode:
                # (requests that bring one row had their state moved on by the kernel above)
                _check(self._ops.distie_conv_state(product, _code(product), W, taps, state,
                                                   meta.cu_q, meta.state_slots, meta.num_requests,
                                                   channels, 1, self._stream()), "conv_state")
            _mark_written(state)
        return q

    def sigmoid_gate(self, x, num_heads, head_stride, width, gates, per_head=False):
        x = self.dense(x)
        self._own(x)
        T = x.shape[0]
        if x.shape[1] != num_heads * head_stride or width > head_stride:
            raise KernelError("sigmoid_gate: x must be [T, heads * head_stride]")
        if per_head:
            if gates is None:
                raise KernelError("sigmoid_gate: a gate for each head needs the gates")
            g_ptr, g_ld = self._rows_view(gates, num_heads)
            out = self._empty((T, num_heads * width), x.dtype)
            _check(self._ops.distie_head_gate(x, _code(x), head_stride, width, g_ptr, _code(gates), g_ld,
                                              out, _code(out), T, num_heads * width, self._stream()), "head_gate")
            return out
        g_ptr, g_ld = self._rows_view(gates, num_heads * width) if gates is not None else (None, 0)
        out = self._empty((T, num_heads * width), x.dtype)
        _check(self._ops.distie_sigmoid_gate(x, _code(x), head_stride, width, g_ptr,
                                             _code(gates) if gates is not None else _code(x), g_ld,
                                             out, _code(out), T, num_heads * width, self._stream()),
               "sigmoid_gate")
        return out

    def _scan_chunks(self, meta, rows, num_heads, dim, value_dim):
        """Which rows of the step form a chunk of a state's scan, worked out from the step's row counts (known on the
        host outside captured steps): (number of chunks, the table {request, first row, rows, 1 for a request that brings one row and
        0 for the others} with the first chunk of every request behind it, scratch for a state a chunk)."""
        table_key = ("scan_chunk_table", rows)
        held = meta.scratch.get(table_key)
        if held is None:
            cu = np.asarray(meta.host_cu_q, dtype=np.int64)
            table, first = [], [0]
            meta.scratch["scan_singles"] = int((cu[1:] - cu[:-1] == 1).sum())
            for b in range(meta.num_requests):
                one = 1 if cu[b + 1] - cu[b] == 1 else 0
                for at in range(int(cu[b]), int(cu[b + 1]), rows):
                    table.append((b, at, min(rows, int(cu[b + 1]) - at), one))
                first.append(len(table))
            packed = self.upload(np.concatenate([np.asarray(table, dtype=np.int32).reshape(-1),
                                                 np.asarray(first, dtype=np.int32)]))
            held = meta.scratch[table_key] = (len(table), packed)
        count, packed = held
        key = ("scan_chunks", rows, num_heads, dim, value_dim)
        scratch = meta.scratch.get(key)
        if scratch is None:
            scratch = meta.scratch[key] = self._empty((count, num_heads, dim, value_dim), torch.float32)
        return count, packed, scratch

    def decay_scan(self, product, state, decay, meta, num_heads, dim, value_dim, act="silu", k_scale=1.0, inv_freq=None,
                   neighbours=False):
        if act not in ("silu", None) or (act is not None and (inv_freq is not None or k_scale != 1.0)):
            raise KernelError("decay_scan: silu on q, k and v, or no activation with a rotation and a scale of k")
        product = self.dense(product)
        self._own(product, state, decay)
        T, W = product.shape
        if T != meta.num_tokens or W < num_heads * (2 * dim + value_dim):
            raise KernelError("decay_scan: the product does not match the batch or the head counts")
        if state.dtype != torch.float32 or tuple(state.shape[1:]) != (num_heads, dim, value_dim):
            raise KernelError("decay_scan: the state is float32 [slots, heads, dim, value_dim]")
        if decay.dtype != torch.float32 or tuple(decay.shape) != (num_heads,):
            raise KernelError("decay_scan: decay must be float32 [heads]")
        if dim > self._ops.distie_decay_scan_max_dim():
            raise KernelError(f"decay_scan: heads of up to {self._ops.distie_decay_scan_max_dim()} dimensions")
        pairs = 0 if inv_freq is None else inv_freq.shape[0]
        if 2 * pairs > dim:
            raise KernelError("decay_scan: the rotation turns more dimensions than a head has")
        table = self._rope_table(meta, inv_freq) if pairs else None
        turn = (1 if act else 0, table.data_ptr() if pairs else None, pairs, 1 if neighbours else 0, float(k_scale))
        out = self._empty((T, num_heads * value_dim), torch.float32)
        if not self.captured and meta.host_cu_q is not None and meta.max_q >= self.SCAN_CHUNKED_MIN_ROWS and \
                dim <= self._ops.distie_decay_scan_chunked_max_dim():
            # portions of prompts: chunks of rows side by side instead of one row after the other. Which rows form
            # a chunk is worked out here from the step's row counts (known on the host outside captured steps).
            count, packed, scratch = self._scan_chunks(meta, self._ops.distie_decay_scan_chunk_rows(), num_heads, dim,
                                                       value_dim)
            _check(self._ops.distie_decay_scan_chunked(
                product, _code(product), W, state, decay, out,
                scratch, packed, packed.data_ptr() + 16 * count, meta.state_slots,
                count, meta.num_requests, num_heads, dim, value_dim, *turn, self._stream()), "decay_scan_chunked")
            _mark_written(state)
            return out
        _check(self._ops.distie_decay_scan(product, _code(product), W, state, decay,
                                           out, meta.cu_q, meta.state_slots,
                                           meta.num_requests, num_heads, dim, value_dim, *turn, self._stream()),
               "decay_scan")
        _mark_written(state)
        return out

    def rmsnorm_gate(self, x, weight, eps, gates, out_dtype, group=None, gate="sigmoid", gate_first=False):
        self._own(x, weight)
        if gate not in ("sigmoid", "silu"):
            raise KernelError(f"rmsnorm_gate: no gate named {gate!r}")
        if gate_first:
            # the gate in front of the norm, every column with a weight of its own
            if gates is None:
                raise KernelError("rmsnorm_gate: no gate to put in front of the norm")
            if x.dtype != torch.float32 or x.dim() != 2 or tuple(weight.shape) != (x.shape[1],) or \
                    (group is not None and (group < 1 or x.shape[1] % group)):
                raise KernelError("rmsnorm_gate: x must be float32 [T, N], weight [N], N a multiple of the group")
            T, N = x.shape
            size = group or N
            g_ptr, g_ld = self._rows_view(gates, N)
            out = self._empty((T, N), out_dtype)
            _check(self._ops.distie_gate_rmsnorm(x, weight, _code(weight), float(eps), g_ptr,
                                                 _code(gates), g_ld, out, _code(out), T, size, N // size,
                                                 1 if gate == "silu" else 0, self._stream()), "gate_rmsnorm")
            return out
        if x.dtype != torch.float32 or x.dim() != 2 or (group is not None and (group < 1 or x.shape[1] % group)) or \
                tuple(weight.shape) not in ((group or x.shape[1],), (x.shape[1],)):
            raise KernelError("rmsnorm_gate: x must be float32 [T, N], weight [N] (or [group], N a multiple of it)")
        T, N = x.shape
        g_ptr, g_ld, g_code = None, 0, _F32
        if gates is not None:
            g_ptr, g_ld = self._rows_view(gates, N)
            g_code = _code(gates)
        out = self._empty((T, N), out_dtype)
        size = group or N
        _check(self._ops.distie_rmsnorm_gate(x, weight, _code(weight), float(eps), g_ptr, g_code,
                                             g_ld, out, _code(out), T, size, N // size,
                                             1 if gate == "silu" else 0, 1 if weight.shape[0] != size else 0,
                                             self._stream()), "rmsnorm_gate")
        return out

    # ---- norms behind sub-layers, mixers side by side, gated states, routers (csrc/recurrent.hip)
    def _term(self, value):
        """(tensor, slices) of a sub-layer's result as the norm kernels read it."""
        if isinstance(value, (NormedSum, PendingNorm, PendingProduct)):
            value = self.dense(value)
        if isinstance(value, PartialSums):
            self._own(value.data)
            return value.data, value.slices
        self._own(value)
        return value, 1

    def _norm_chain(self, terms, weights, term_eps, scale, post, residual, pre, out_dtype):
        held = [self._term(t) for t in terms]
        T, C = held[0][0].shape[-2:]
        for tensor, _ in held:
            if tuple(tensor.shape[-2:]) != (T, C):
                raise KernelError("norm chain: the terms must all be [T, C]")
        vectors = list(weights or []) + [v[0] for v in (post, pre) if v is not None]
        self._own(*vectors)
        for w in vectors:
            if w.dtype != torch.float32 or tuple(w.shape) != (C,):
                raise KernelError("norm chain: norm weights are float32 [C]")
        if residual is not None:
            self._own(residual)
            if residual.dtype != torch.float32 or tuple(residual.shape) != (T, C):
                raise KernelError("norm chain: the residual is float32 [T, C]")
        out = y = None
        if residual is None:
            y = self._empty((T, C), torch.float32)
        elif out_dtype is not None:
            # with a norm in front of the next sub-layer (`pre`), or the new residual as it is, in `out_dtype`
            out = self._empty((T, C), out_dtype)
        (t0, s0), (t1, s1) = held[0], (held[1] if len(held) > 1 else (None, 1))
        _check(self._ops.distie_norm_chain(
            t0, _code(t0), s0, weights[0] if weights else None, t1, _code(t1) if t1 is not None else _F32,
            s1, weights[1] if weights and len(weights) > 1 else None, float(term_eps), float(scale),
            post[0] if post else None, float(post[1]) if post else 0.0, residual,
            pre[0] if pre else None, float(pre[1]) if pre else 0.0, out, _code(out) if out is not None else _F32,
            y, T, C, self._stream()), "norm_chain")
        if residual is not None:
            _mark_written(residual)
        return out if residual is not None else y

    def normed_sum(self, terms, weights, eps, scale):
        if not 1 <= len(terms) <= 2 or len(weights) != len(terms):
            raise KernelError("normed_sum takes one or two terms, a weight for each")
        return NormedSum(list(terms), [self._f32(w) for w in weights], float(eps), float(scale))

    @staticmethod
    def _f32(weight):
        """A norm's weight as float32 (a bfloat16 value is one exactly); kept on the tensor."""
        if weight.dtype == torch.float32:
            return weight
        held = getattr(weight, "_distie_f32", None)
        if held is None:
            held = weight._distie_f32 = weight.float()
        return held

    def add_normed(self, residual, delta, weight, eps):
        self.add_normed_rmsnorm(residual, delta, weight, eps, None, 0.0, None)

    def add_normed_rmsnorm(self, residual, delta, post_weight, post_eps, weight, eps, out_dtype):
        post = (self._f32(post_weight), post_eps)
        pre = (self._f32(weight), eps) if weight is not None else None
        if isinstance(delta, NormedSum):
            return self._norm_chain(delta.terms, delta.weights, delta.eps, delta.scale, post, residual, pre, out_dtype)
        return self._norm_chain([delta], None, 0.0, 1.0, post, residual, pre, out_dtype)

    def read_residual(self, residual, out_dtype):
        self._own(residual)
        if residual.dtype != torch.float32 or residual.dim() != 2:
            raise KernelError("read_residual reads the float32 residual stream")
        if out_dtype == torch.float32:
            return residual
        out = self._empty(residual.shape, out_dtype)
        _check(self._ops.distie_sum_slices(residual, 1, out.numel(), out, _CODES[out_dtype],
                                           self._stream()), "sum_slices")
        return out

    def add_normed_read(self, residual, delta, post_weight, post_eps, out_dtype):
        if out_dtype == torch.float32:
            self.add_normed(residual, delta, post_weight, post_eps)
            return residual
        post = (self._f32(post_weight), post_eps)
        if isinstance(delta, NormedSum):
            return self._norm_chain(delta.terms, delta.weights, delta.eps, delta.scale, post, residual, None, out_dtype)
        return self._norm_chain([delta], None, 0.0, 1.0, post, residual, None, out_dtype)

    def gated_decay_scan(self, product, decay_logits, state, meta, num_heads, dim, value_dim, q_scale, tau, decay_low=None):
        product = self.dense(product)
        self._own(product, decay_logits, state)
        T, W = product.shape
        if T != meta.num_tokens or W < num_heads * (2 * dim + value_dim):
            raise KernelError("gated_decay_scan: the product does not match the batch or the head counts")
        if state.dtype != torch.float32 or tuple(state.shape[1:]) != (num_heads, dim, value_dim):
            raise KernelError("gated_decay_scan: the state is float32 [slots, heads, dim, value_dim]")
        chunked = not self.captured and meta.host_cu_q is not None and meta.max_q >= self.SCAN_CHUNKED_MIN_ROWS and \
            dim % 4 == 0 and value_dim % 4 == 0 and dim <= self._ops.distie_gated_decay_scan_chunked_max_dim()
        low_ptr, low_ld, up, up_bias, rank = None, 0, None, None, 0
        if decay_logits is None:
            if decay_low is None:
                raise KernelError("gated_decay_scan: neither the decay's logits nor what they are made from")
            low, up, up_bias = decay_low
            rank = up.shape[1]
            if tuple(up.shape) != (num_heads * dim, rank) or low.shape[0] != T or low.dtype != product.dtype or \
                    up_bias.dtype != torch.float32 or tuple(up_bias.shape) != (num_heads * dim,):
                raise KernelError("gated_decay_scan: low [T, rank] of the product's dtype, up [heads * dim, rank], "
                                  "bias float32 [heads * dim]")
            if chunked or rank > self._ops.distie_gated_decay_scan_max_rank():
                # portions of prompts (and wide projections): the logits as a product of their own
                decay_logits = self.decay_logits_of(decay_low)
            else:
                low_ptr, low_ld = self._rows_view(low, rank)
                up = self._f32(up)
                self._own(up, up_bias)
        if decay_logits is not None and (decay_logits.dtype != torch.float32 or
                                         tuple(decay_logits.shape) != (T, num_heads * dim)):
            raise KernelError("gated_decay_scan: the decay's logits are float32 [T, heads * dim]")
        out = self._empty((T, num_heads * value_dim), torch.float32)
        if chunked:
            # portions of prompts: chunks of rows side by side instead of one row after the other
            count, packed, scratch = self._scan_chunks(meta, self._ops.distie_gated_decay_scan_chunk_rows(), num_heads,
                                                       dim, value_dim)
            totals = self._empty((count, num_heads, dim), torch.float32)
            _check(self._ops.distie_gated_decay_scan_chunked(
                product, _code(product), W, decay_logits, state, out,
                scratch, totals, packed, packed.data_ptr() + 16 * count,
                meta.state_slots, count, meta.num_requests, num_heads, dim, value_dim, float(q_scale),
                float(tau), self._stream()), "gated_decay_scan_chunked")
            _mark_written(state)
            return out
        _check(self._ops.distie_gated_decay_scan(
            product, _code(product), W, decay_logits,
            low_ptr, low_ld, up if low_ptr is not None else None,
            up_bias if low_ptr is not None else None, rank if low_ptr is not None else 0, state,
            out, meta.cu_q, meta.state_slots, meta.num_requests, num_heads, dim,
            value_dim, float(q_scale), float(tau), self._stream()), "gated_decay_scan")
        _mark_written(state)
        return out

    # ---- time mixing with a token shift, norms in groups, averages over the depth (csrc/time_mixing.hip, csrc/depth.hip)
    def token_shift(self, x, mu, state, meta):
        x = self.dense(x)
        self._own(x, mu, state)
        T, C = x.shape
        if T != meta.num_tokens or mu.dtype != torch.float32 or mu.dim() != 2 or mu.shape[1] != C:
            raise KernelError("token_shift: x are the step's rows, mu float32 [mixes, C]")
        if state.dtype != torch.float32 or tuple(state.shape[1:]) != (C,):
            raise KernelError("token_shift: the state is float32 [slots, C]")
        out = self._empty((mu.shape[0], T, C), x.dtype)
        _check(self._ops.distie_token_shift(x, _code(x), mu, mu.shape[0], state,
                                            out, meta.cu_q, None if meta.all_decode else meta.token_request,
                                            meta.state_slots, T, C, self._stream()), "token_shift")
        _mark_written(state)
        return out

    EACH_MAX_ROWS = 32        # up to so many rows several products with inputs of their own run in the kernel for few rows

    def prepare_linear_each(self, weights):
        """One packed copy for all, kept on the first weight: the weights one behind the other, each rounded up to whole
        row blocks. Up to EACH_MAX_ROWS rows all products share a launch of the kernel for few rows; of more rows the rounded ones
        share one of the large tiles, and the library takes the unrounded one and what is beyond LARGE_EACH_WORK."""
        first = weights[0]
        if (self.packed_roles is not None and "qkv" not in self.packed_roles) or not self.packed_weights or \
                any(w.dtype != torch.bfloat16 or w.dim() != 2 or w.shape[1] != first.shape[1] for w in weights) or \
                first.shape[1] % 8 or len(weights) > 8 or hasattr(first, "_distie_each"):
            return
        K = first.shape[1]
        blocks = [-(-w.shape[0] // 16) for w in weights]
        free, total = torch.cuda.mem_get_info(self.device)
        if free - 2 * sum(blocks) * -(-K // 32) * 512 < self.PACKED_KEEPS_FREE * total:
            self._packed_left_out += 1
            return
        packed = self._empty(sum(blocks) * -(-K // 32) * 512, torch.bfloat16)
        at, maps = 0, []
        for w, count in zip(weights, blocks):
            self._own(w)
            row_map = self._row_map(w.shape[0], False, None).to(device=self.device, dtype=torch.int32)
            maps.append(row_map)
            size = count * -(-K // 32) * 512
            _check(self._ops.distie_pack_rows(w, packed[at:at + size], row_map, count, K,
                                              self._stream()), "pack_rows")
            at += size
        torch.cuda.current_stream(self.device).synchronize()      # the row maps are freed on return
        first._distie_each = (packed, np.cumsum(np.asarray(blocks, dtype=np.int32)).astype(np.int32))

    def linear_each(self, xs, weights, unrounded=()):
        held = getattr(weights[0], "_distie_each", None)
        if held is None or xs.dtype != torch.bfloat16:
            return super().linear_each(xs, weights, unrounded)
        packed, ends = held
        count, M, K = xs.shape
        plan = None
        if M > self.EACH_MAX_ROWS:
            # the rounded ones in one launch, if they are the first; the others one by one
            rounded = count - len(unrounded)
            if rounded > 1 and all(k >= rounded for k in unrounded):
                plan = self._large_each(M, 16 * int(ends[rounded - 1]), K, xs)
            if plan is None:
                return super().linear_each(xs, weights, unrounded)
        self._own(xs)
        if count != len(weights) or any(w.shape[1] != K for w in weights) or \
                [int(e) for e in np.diff(ends, prepend=0)] != [-(-w.shape[0] // 16) for w in weights] or \
                packed.numel() != int(ends[-1]) * -(-K // 32) * 512:
            raise KernelError("linear_each: an input [rows, K] for every weight [N, K], the weights it was prepared for")
        starts = [0] + [16 * int(e) for e in ends[:-1]]
        if plan is not None:
            out = self._empty((M, 16 * int(ends[rounded - 1])), torch.bfloat16)
            _check(self._ops.distie_large_tiles_each_bf16(xs, packed, out, M, K, rounded,
                                                          ends.ctypes.data, plan, self._stream()), "large_tiles_each_bf16")
            return [out[:, at:at + w.shape[0]] for at, w in zip(starts, weights[:rounded])] + \
                [self.linear_f32out(xs[k], weights[k]) for k in range(rounded, count)]
        out = self._empty((M, 16 * int(ends[-1])), torch.float32)
        _check(self._ops.distie_gemm_packed_each_bf16(xs, packed, out, M, K, count,
                                                      ends.ctypes.data, self._stream()), "gemm_packed_each_bf16")
        return [out[:, at:at + w.shape[0]] for at, w in zip(starts, weights)]

    def wkv_decay_logits(self, low, up, up_bias):
        low = low if low.dtype == torch.float32 else low.float()
        ptr, ld = self._rows_view(low, up.shape[1])
        bent = self._empty(low.shape, torch.float32)
        _check(self._ops.distie_tanh_f32(ptr, ld, bent, low.shape[0], low.shape[1], self._stream()), "tanh_f32")
        return self.linear_f32out(bent, up, up_bias)

    def wkv_mix(self, r, k, v, gates, low, up, up_bias, bonus, state, meta, num_heads, dim, norm_weight, eps, out_dtype):
        N, T, rank = num_heads * dim, r.shape[0], up.shape[1]
        self._own(up, up_bias, bonus, state, norm_weight)
        views = [self._rows_view(t, N) for t in (r, k, v, gates)]
        ld = views[0][1]
        if T != meta.num_tokens or any(t.dtype != r.dtype or t.shape[0] != T for t in (k, v, gates)) or \
                any(view[1] != ld for view in views) or low.shape[0] != T:
            raise KernelError("wkv_mix: r, k, v and gates are the step's rows, of one dtype and row stride")
        for name, t, shape in (("up", up, (N, rank)), ("up_bias", up_bias, (N,)), ("bonus", bonus, (N,)),
                               ("norm_weight", norm_weight, (N,))):
            if t.dtype != torch.float32 or tuple(t.shape) != shape:
                raise KernelError(f"wkv_mix: {name} must be float32 {list(shape)}")
        if state.dtype != torch.float32 or tuple(state.shape[1:]) != (num_heads, dim, dim):
            raise KernelError("wkv_mix: the state is float32 [slots, heads, dim, dim]")
        if dim > self._ops.distie_wkv_scan_max_dim() or rank > self._ops.distie_wkv_scan_max_rank():
            raise KernelError(f"wkv_mix: heads of up to {self._ops.distie_wkv_scan_max_dim()} and decays through up to "
                              f"{self._ops.distie_wkv_scan_max_rank()} dimensions")
        low_ptr, low_ld = self._rows_view(low, rank)
        out = self._empty((T, N), out_dtype)
        if not self.captured and meta.host_cu_q is not None and meta.max_q >= self.SCAN_CHUNKED_MIN_ROWS and \
                dim <= self._ops.distie_wkv_chunked_max_dim():
            # portions of prompts: chunks of rows side by side instead of one row after the other
            z = self.wkv_decay_logits(low, up, up_bias)
            count, packed, scratch = self._scan_chunks(meta, self._ops.distie_wkv_chunk_rows(), num_heads, dim, dim)
            totals = self._empty((count, num_heads, dim), torch.float32)
            _check(self._ops.distie_wkv_scan_chunked(
                views[0][0], views[1][0], views[2][0], views[3][0], _code(r), ld, z, bonus,
                state, norm_weight, float(eps), out, _code(out), scratch,
                totals, packed, packed.data_ptr() + 16 * count, meta.state_slots, count,
                meta.num_requests, num_heads, dim, self._stream()), "wkv_scan_chunked")
            _mark_written(state)
            return out
        _check(self._ops.distie_wkv_scan(
            views[0][0], views[1][0], views[2][0], views[3][0], _code(r), ld, low_ptr, _code(low), low_ld, rank, up,
            up_bias, bonus, state, norm_weight, float(eps), out,
            _code(out), None if meta.all_decode else meta.cu_q, meta.state_slots, meta.num_requests,
            num_heads, dim, self._stream()), "wkv_scan")
        _mark_written(state)
        return out

    def group_rmsnorm(self, x, weight, eps, groups, out_dtype):
        return self._group_chain(x, weight, eps, groups, None, None, None, out_dtype)

    def _group_chain(self, delta, weight, eps, groups, residual, into, history, out_dtype, shift=None):
        delta, slices = self._term(delta)
        T, C = delta.shape[-2:]
        self._own(weight, residual, into)
        if weight.dtype != torch.float32 or tuple(weight.shape) != (C,) or groups < 1 or C % groups:
            raise KernelError("norm in groups: weight float32 [C], C a multiple of the groups")
        for t in (residual, into):
            if t is not None and (t.dtype != torch.float32 or tuple(t.shape) != (T, C)):
                raise KernelError("norm in groups: the residual is float32 [T, C]")
        first = rest = weights = None
        index = 0
        if history is not None:
            first, rest, index, weights = history
            self._own(first, rest, weights)
            if first.dtype != torch.float32 or rest.dtype != torch.float32 or tuple(first.shape) != (T, C) or \
                    rest.dim() != 3 or tuple(rest.shape[1:]) != (T, C) or not 0 <= index < rest.shape[0] or \
                    weights.dtype != torch.float32 or tuple(weights.shape) != (index + 2,):
                raise KernelError("average over the depth: X_0 float32 [T, C], the others [layers, T, C], a weight for each")
        mu = state = slots = None
        if shift is not None:
            mu, state, slots = shift
            self._own(mu, state, slots)
            if mu.dtype != torch.float32 or mu.dim() != 2 or mu.shape[1] != C or slots.shape[0] != T or \
                    state.dtype != torch.float32 or tuple(state.shape[1:]) != (C,):
                raise KernelError("norm in groups with a token shift: mu float32 [mixes, C], the state float32 [slots, C], a row "
                                  "a request")
        out = None
        if out_dtype is not None:
            out = self._empty((T, C) if mu is None else (mu.shape[0], T, C), out_dtype)
        _check(self._ops.distie_group_chain(
            delta, _code(delta), slices, weight, float(eps), int(groups), residual, into,
            first, rest, int(index), weights, out, _code(out) if out is not None else _F32, T, C, mu,
            mu.shape[0] if mu is not None else 0, state, slots, self._stream()), "group_chain")
        if state is not None:
            _mark_written(state)
        if into is not None:
            _mark_written(into)
        return out

    def add_group_normed(self, residual, delta, weight, eps, groups, out_dtype, in_place=True, history=None):
        into = residual if in_place else torch.empty_like(residual)
        read = self._group_chain(delta, weight, eps, groups, residual, into, history,
                                 None if out_dtype == torch.float32 else out_dtype)
        return into, into if out_dtype == torch.float32 else read

    def add_group_normed_shift(self, residual, delta, weight, eps, groups, out_dtype, in_place, history, mu, state, meta):
        if not meta.all_decode:
            return super().add_group_normed_shift(residual, delta, weight, eps, groups, out_dtype, in_place, history, mu, state,
                                                  meta)
        # a row a request: the block that owns a row shifts it too
        into = residual if in_place else torch.empty_like(residual)
        return into, self._group_chain(delta, weight, eps, groups, residual, into, history, out_dtype,
                                       (mu, state, meta.state_slots))

    def lru_gates(self, u, recur_weight, recur_bias, input_weight, input_bias, lam, rate):
        u = self.dense(u)
        self._own(recur_weight, recur_bias, input_weight, input_bias, lam)
        T, R = u.shape
        u_ptr, ldu = self._rows_view(u, R)
        blocks = recur_weight.shape[0]
        n = R // max(blocks, 1)
        if recur_weight.dim() != 3 or tuple(recur_weight.shape) != (blocks, n, n) or blocks * n != R or \
                input_weight.shape != recur_weight.shape or input_weight.dtype != recur_weight.dtype:
            raise KernelError("lru_gates: the gates' weights are [blocks, R / blocks, R / blocks], of one dtype")
        for t in (recur_bias, input_bias, lam):
            if t.dtype != torch.float32 or t.numel() != R:
                raise KernelError("lru_gates: biases and lam are float32 with R elements")
        a = self._empty((T, R), torch.float32)
        x = self._empty((T, R), torch.float32)
        _check(self._ops.distie_lru_gates(u_ptr, _code(u), ldu, recur_weight, recur_bias,
                                          input_weight, input_bias, _code(recur_weight),
                                          lam, float(rate), a, x, T, R, blocks,
                                          self._stream()), "lru_gates")
        return a, x

    def lru_scan(self, a, x, state, meta, mul, mul_act, out_dtype):
        self._own(a, x, state)
        T, R = a.shape
        if a.dtype != torch.float32 or x.dtype != torch.float32 or x.shape != a.shape or T != meta.num_tokens:
            raise KernelError("lru_scan: a and x are float32 [T, R], the step's rows")
        if state.dtype != torch.float32 or tuple(state.shape[1:]) != (R,):
            raise KernelError("lru_scan: the state is float32 [slots, R]")
        kind = -1
        if mul_act is not None:
            if mul_act not in self.ACTIVATIONS:
                raise KernelError(f"no activation named {mul_act!r}")
            kind = self.ACTIVATIONS[mul_act]
        m_ptr, m_ld, m_code = None, 0, _F32
        if mul is not None:
            m_ptr, m_ld = self._rows_view(mul, R)
            m_code = _code(mul)
        out = self._empty((T, R), out_dtype)
        if not self.captured and meta.host_cu_q is not None and meta.max_q >= self.LRU_CHUNKED_MIN_ROWS:
            # portions of prompts: chunks of rows side by side, each scanned twice (alone, then from what stands before it)
            count, packed, sums = self._scan_chunks(meta, self._ops.distie_lru_scan_chunk_rows(), 1, 1, R)
            factors = self._empty((count, R), torch.float32)
            init = self._empty((meta.num_requests, R), torch.float32)
            _check(self._ops.distie_lru_scan_chunked(
                a, x, state, factors, sums, init, m_ptr,
                m_code, m_ld, kind, out, _code(out), packed, packed.data_ptr() + 16 * count,
                meta.state_slots, count, meta.num_requests, R, self._stream()), "lru_scan_chunked")
            _mark_written(state)
            return out
        _check(self._ops.distie_lru_scan(a, x, state, m_ptr, m_code, m_ld, kind,
                                         out, _code(out), meta.cu_q, meta.state_slots,
                                         meta.num_requests, R, self._stream()), "lru_scan")
        _mark_written(state)
        return out

    SCORINGS = {"softmax": 0, "sigmoid": 1, "softmax_all": 2, "sigmoid_share": 3}
    NO_RULE = RouteRule()

    def _route_rule(self, rule, scoring, experts):
        """The rule's numbers as the kernels take them: (correction, groups, kept, scale, shared)."""
        rule = rule or self.NO_RULE
        if scoring != "sigmoid_share" and (rule.correction is not None or rule.groups != 1 or rule.scale != 1.0):
            raise KernelError("a router's correction, groups and scale go with the scoring sigmoid_share")
        self._own(rule.correction)
        if rule.correction is not None and (rule.correction.dtype != torch.float32 or tuple(rule.correction.shape) != (experts,)):
            raise KernelError("a router's correction is float32 [experts]")
        return (rule.correction.data_ptr() if rule.correction is not None else None, int(rule.groups), int(rule.kept),
                float(rule.scale), 1 if rule.shared else 0)

    def route_topk(self, x, weight, bias, top, scoring="softmax", rule=None):
        if scoring not in self.SCORINGS:
            raise KernelError(f"route_topk: no scoring named {scoring!r}")
        x = self.dense(x)
        self._own(x, weight, bias)
        T, C = x.shape
        rows = weight.shape[0]
        shared = 1 if rule is not None and rule.shared else 0
        E = rows - shared
        if tuple(weight.shape) != (rows, C) or (bias is not None and (bias.dtype != torch.float32 or tuple(bias.shape) != (rows,))):
            raise KernelError("route_topk: weight [experts (+ 1 with a shared one), C], bias float32 with a number a row")
        numbers = self._route_rule(rule, scoring, E)
        experts = self._empty((T, top), torch.int32)
        gates = self._empty((T, top + shared), torch.float32)
        _check(self._ops.distie_route_topk(x, _code(x), weight, _code(weight),
                                           bias, experts,
                                           gates, T, C, E, int(top), self.SCORINGS[scoring], *numbers,
                                           self._stream()), "route_topk")
        return experts, gates

    def route_glu(self, gate_up, experts, gates, num_experts, width, limit, slope, up_shift, on_input, shared_width=0):
        if isinstance(gate_up, (PendingNorm, PendingProduct)):
            gate_up = self.dense(gate_up)
        slices, source, dtype, ld = 1, gate_up, gate_up.dtype, gate_up.shape[1]
        if isinstance(gate_up, PartialSums):
            slices, source = gate_up.slices, gate_up.data
        elif gate_up.dim() == 2 and gate_up.stride(1) == 1 and gate_up.stride(0) > gate_up.shape[1]:
            # rows that lie further apart than they are wide (`linear_spread`): the kernel takes the row stride
            ld = gate_up.stride(0)
            if gate_up.device != self.device:
                raise KernelError(f"tensor on {gate_up.device}, kernels run on {self.device}")
            source = None
        self._own(source, experts, gates)
        source = gate_up if source is None else source
        T, top = experts.shape
        total = num_experts * width + shared_width
        if experts.dtype != torch.int32 or gates.dtype != torch.float32 or \
                tuple(gates.shape) != (T, top + (1 if shared_width else 0)) or \
                gate_up.shape[0] != T or gate_up.shape[1] != 2 * total:
            raise KernelError("route_glu: experts int32 and gates float32 [T, top] (one more with a shared expert), gate_up "
                              "[T, 2 * (experts * width + shared_width)]")
        if limit is not None and not limit > 0:
            raise KernelError("route_glu: the limit must be positive")
        out = self._empty((T, total), dtype)
        _check(self._ops.distie_route_glu(source, _code(source), ld, slices, experts,
                                          gates, T, top, num_experts, width, float(limit or 0.0), float(slope),
                                          float(up_shift), 1 if on_input else 0, int(shared_width), out,
                                          _code(out), self._stream()), "route_glu")
        return out

    FUSED_ROUTE_ROWS = 64       # up to so many rows every block works out its row's choice itself

    def route_experts_glu(self, x, router_weight, router_bias, top, scoring, gate_up, num_experts, width, limit, slope,
                          up_shift, on_input, rule=None, shared_width=0):
        if scoring not in self.SCORINGS:
            raise KernelError(f"route_experts_glu: no scoring named {scoring!r}")
        x = self.dense(x)
        T, C = x.shape
        if T > self.FUSED_ROUTE_ROWS or x.dtype != torch.bfloat16 or router_weight.dtype != torch.bfloat16 or C % 8 or \
                x.data_ptr() % 16 or router_weight.data_ptr() % 16 or not x.is_contiguous():
            return super().route_experts_glu(x, router_weight, router_bias, top, scoring, gate_up, num_experts, width,
                                             limit, slope, up_shift, on_input, rule, shared_width)
        if isinstance(gate_up, (PendingNorm, PendingProduct)):
            gate_up = self.dense(gate_up)
        slices, source, dtype = 1, gate_up, gate_up.dtype
        if isinstance(gate_up, PartialSums):
            slices, source = gate_up.slices, gate_up.data
        self._own(x, router_weight, router_bias, source)
        numbers = self._route_rule(rule, scoring, num_experts)
        rows, total = num_experts + numbers[-1], num_experts * width + shared_width
        if tuple(router_weight.shape) != (rows, C) or not 1 <= top <= num_experts or gate_up.shape[0] != T or \
                gate_up.shape[1] != 2 * total or (shared_width and not numbers[-1]) or \
                (router_bias is not None and (router_bias.dtype != torch.float32 or tuple(router_bias.shape) != (rows,))):
            raise KernelError("route_experts_glu: x [T, C], router [E, C], bias float32 [E], gate_up [T, 2 * E * width]")
        if limit is not None and not limit > 0:
            raise KernelError("route_experts_glu: the limit must be positive")
        out = self._empty((T, total), dtype)
        _check(self._ops.distie_route_topk_glu(
            x, router_weight, router_bias, C,
            self.SCORINGS[scoring], source, _code(source), gate_up.shape[1], slices, T, int(top),
            num_experts, width, float(limit or 0.0), float(slope), float(up_shift), 1 if on_input else 0, *numbers,
            int(shared_width), out, _code(out), self._stream()), "route_topk_glu")
        return out

    def softcap(self, x, cap):
        self._own(x)
        if x.dtype != torch.float32:
            raise KernelError("softcap works on float32 values")
        _check(self._ops.distie_softcap_f32(x, x.numel(), float(cap), self._stream()), "softcap_f32")
        _mark_written(x)
        return x

    def route_scale(self, hidden, experts, gates, num_experts, width):
        hidden = self.dense(hidden)
        self._own(hidden, experts, gates)
        T, top = experts.shape
        if experts.dtype != torch.int32 or gates.dtype != torch.float32 or gates.shape != experts.shape or \
                hidden.shape[0] != T or hidden.shape[1] < num_experts * width:
            raise KernelError("route_scale: experts int32 and gates float32 [T, top], hidden [T, >= experts * width]")
        _check(self._ops.distie_route_scale(hidden, _code(hidden), hidden.shape[1], experts,
                                            gates, T, top, num_experts, width, self._stream()), "route_scale")
        _mark_written(hidden)
        return hidden

    def activation(self, x, kind):
        if kind not in self.ACTIVATIONS:
            raise KernelError(f"no activation named {kind!r}")
        if isinstance(x, (PendingNorm, PendingProduct)):
            x = self.dense(x)
        slices, source, dtype = 1, x, x.dtype
        if isinstance(x, PartialSums):
            slices, source = x.slices, x.data
        self._own(source)
        out = self._empty(tuple(x.shape), dtype)
        _check(self._ops.distie_activation(source, _code(source), slices, out, _code(out), out.numel(),
                                           self.ACTIVATIONS[kind], self._stream()), "activation")
        return out

    # ---- the gated delta rule (csrc/delta.hip)
    def delta_scan(self, qkv, beta, decay, a_log, dt_bias, state, meta, num_heads, num_kv_heads, dim, value_dim, q_scale,
                   unit_eps):
        qkv = self.dense(qkv)
        H, G, D, E = num_heads, num_kv_heads, dim, value_dim
        q_ptr, ld = self._rows_view(qkv, qkv.shape[1])
        b_ptr, ldb = self._rows_view(beta, H)
        d_ptr, ldd = self._rows_view(decay, H)
        self._own(a_log, dt_bias, state)
        T = qkv.shape[0]
        if T != meta.num_tokens or qkv.shape[1] < 2 * G * D + H * E or H % G or beta.shape[0] != T or decay.shape[0] != T or \
                beta.dtype != qkv.dtype or decay.dtype != qkv.dtype:
            raise KernelError("delta_scan: q, k, v and the logits do not match the batch or the head counts")
        if D > self._ops.distie_delta_scan_max_dim():
            raise KernelError(f"delta_scan: keys of up to {self._ops.distie_delta_scan_max_dim()} dimensions a head")
        if state.dtype != torch.float32 or tuple(state.shape[1:]) != (H, D, E):
            raise KernelError("delta_scan: the state is float32 [slots, heads, dim, value_dim]")
        for vector in (a_log, dt_bias):
            if vector.dtype != torch.float32 or tuple(vector.shape) != (H,):
                raise KernelError("delta_scan: a_log and dt_bias are float32 [heads]")
        out = self._empty((T, H * E), torch.float32)
        if not self.captured and meta.host_cu_q is not None and meta.max_q >= self.SCAN_CHUNKED_MIN_ROWS:
            # portions of prompts: chunks of rows, the triangular systems of all chunks side by side
            rows = self._ops.distie_delta_scan_chunk_rows()
            DP, EP = self._ops.distie_delta_scan_padded_dim(D), -(-E // 16) * 16
            count, packed, states = self._scan_chunks(meta, rows, H, DP, EP)
            key = ("delta_scratch", count, H, DP, EP)
            held = meta.scratch.get(key)
            if held is None:
                held = meta.scratch[key] = [self._empty((count, H, *shape), torch.float32)
                                            for shape in ((rows, DP), (rows, EP), (rows, EP), (DP, rows), (rows, rows), (rows,),
                                                          ())]
            _check(self._ops.distie_delta_scan_chunked(
                q_ptr, _code(qkv), ld, b_ptr, ldb, d_ptr, ldd, a_log, dt_bias, state,
                out, *(t for t in held), states, packed,
                packed.data_ptr() + 16 * count, meta.state_slots, count, meta.num_requests, H, G, D, E,
                float(q_scale), float(unit_eps), self._stream()), "delta_scan_chunked")
            _mark_written(state)
            return out
        _check(self._ops.distie_delta_scan(
            q_ptr, _code(qkv), ld, b_ptr, ldb, d_ptr, ldd, a_log, dt_bias, state,
            out, meta.cu_q, meta.state_slots, meta.num_requests, H, G, D, E, float(q_scale),
            float(unit_eps), self._stream()), "delta_scan")
        _mark_written(state)
        return out

    # ---- a state with one decay a head and token, attention over a shared latent (csrc/ssm.hip, csrc/latent.hip)
    SSM_CHUNKED_MIN_ROWS = 32        # a step with a portion of so many rows scans the state-space state in chunks

    def ssm_scan_captures(self, state_size):
        return state_size <= self._ops.distie_ssm_scan_max_state()

    def ssm_scan(self, xbc, dt, dt_bias, a_log, skip, state, meta, num_heads, value_dim, state_size, groups):
        xbc = self.dense(xbc)
        H, P, N, G = num_heads, value_dim, state_size, groups
        width = H * P + 2 * G * N
        x_ptr, ld = self._rows_view(xbc, xbc.shape[1])
        d_ptr, ldd = self._rows_view(dt, H)
        self._own(dt_bias, a_log, skip, state)
        T = xbc.shape[0]
        if T != meta.num_tokens or xbc.shape[1] < width or dt.dtype != xbc.dtype or H % G:
            raise KernelError("ssm_scan: x, B and C do not match the batch or the head counts")
        if state.dtype != torch.float32 or tuple(state.shape[1:]) != (H, N, P):
            raise KernelError("ssm_scan: the state is float32 [slots, heads, state_size, value_dim]")
        for vector in (dt_bias, a_log, skip):
            if vector.dtype != torch.float32 or tuple(vector.shape) != (H,):
                raise KernelError("ssm_scan: dt_bias, a_log and skip are float32 [heads]")
        out = self._empty((T, H * P), torch.float32)
        wide = N > self._ops.distie_ssm_scan_max_state()      # more rows a head than the row-by-row kernel keeps
        if not self.captured and meta.host_cu_q is not None and (meta.max_q >= self.SSM_CHUNKED_MIN_ROWS or wide):
            count, packed, scratch = self._scan_chunks(meta, self._ops.distie_ssm_scan_chunk_rows(), H, N, P)
            key = ("ssm_totals", count, H, G)
            held = meta.scratch.get(key)
            if held is None:
                rows = self._ops.distie_ssm_scan_chunk_rows()
                held = meta.scratch[key] = (self._empty((count, H), torch.float32),
                                            self._empty((count, G, rows, rows), torch.float32))
            totals, pairs = held
            _check(self._ops.distie_ssm_scan_chunked(
                x_ptr, _code(xbc), ld, d_ptr, ldd, dt_bias, a_log, skip,
                state, out, scratch, totals, pairs, packed,
                packed.data_ptr() + 16 * count, meta.cu_q, meta.state_slots, count, meta.num_requests,
                meta.scratch["scan_singles"], H, P, N, G, self._stream()), "ssm_scan_chunked")
            _mark_written(state)
            return out
        if wide:
            raise KernelError(f"ssm_scan: a state of {N} rows a head is beyond the row-by-row kernel, which is all a "
                              f"captured step can use")
        _check(self._ops.distie_ssm_scan(x_ptr, _code(xbc), ld, d_ptr, ldd, dt_bias, a_log,
                                         skip, state, out, meta.cu_q,
                                         meta.state_slots, meta.num_requests, H, P, N, G, self._stream()),
               "ssm_scan")
        _mark_written(state)
        return out

    def latent_norm_rope_write(self, down, q_rank, q_weight, kv_rank, kv_weight, eps, rot_dim, inv_freq, magnitude,
                               neighbours, meta, group, k_cache, v_cache, write, out_dtype):
        slices = 1
        if isinstance(down, PartialSums) and down.dtype == torch.float32 and \
                down.shape[1] <= self._ops.distie_latent_norm_max_width():
            slices, down = down.slices, down.data.view(-1, down.data.shape[-1])        # added up while they are read
        else:
            down = self.dense(down)
        self._own(down, q_weight, kv_weight, k_cache, v_cache, inv_freq)
        T, W = down.shape[0] // slices, down.shape[1]
        if slices == 1 and W > self._ops.distie_latent_norm_max_width():
            raise KernelError("latent_norm_rope_write: the down-projection is wider than the kernel's row")
        if down.dtype != torch.float32 or W < q_rank + kv_rank + rot_dim or T != meta.num_tokens:
            raise KernelError("latent_norm_rope_write: the down-projection is float32 [T, q_rank + kv_rank + rot_dim]")
        for weight, size in ((q_weight, q_rank), (kv_weight, kv_rank)):
            if size and (weight is None or weight.dtype != torch.float32 or tuple(weight.shape) != (size,)):
                raise KernelError("latent_norm_rope_write: the norms' weights are float32 [rank]")
        padded = k_cache.shape[-1]
        if write:
            self._check_cache(k_cache, v_cache, 1, meta.block_size, padded)
            if k_cache.dtype != v_cache.dtype or padded < kv_rank + rot_dim:
                raise KernelError("latent_norm_rope_write: one key/value head of at least kv_rank + rot_dim, in one dtype")
        pairs = 0 if inv_freq is None else inv_freq.shape[0]
        if pairs and 2 * pairs != rot_dim:
            raise KernelError("latent_norm_rope_write: the rotation turns all of the rotated part")
        table = self._rope_table(meta, inv_freq) if pairs else None
        latent = self._empty((T, q_rank), out_dtype) if q_rank else None
        _check(self._ops.distie_latent_norm_rope_write(
            down, slices, W, q_rank, q_weight, kv_rank, kv_weight, float(eps), rot_dim, table,
            float(magnitude), 1 if neighbours else 0, latent, _CODES[out_dtype], k_cache,
            v_cache, _code(k_cache), meta.groups[group].slots, T, meta.block_size, padded,
            1 if write else 0, self._stream()), "latent_norm_rope_write")
        return latent

    def latent_queries(self, q, key_up, num_heads, dim, rot_dim, padded_dim, inv_freq, magnitude, neighbours, meta):
        """One launch on the matrix cores for bfloat16 steps (the product's partial sums added up while they are read);
        else the product by head, then the rotation."""
        kv_rank = key_up.shape[1]
        slices, source, dtype = 1, q, getattr(q, "dtype", None)
        if isinstance(q, PartialSums):
            slices, source = q.slices, q.data
        fused = dtype == torch.bfloat16 and key_up.dtype == torch.bfloat16 and inv_freq is not None and \
            isinstance(source, torch.Tensor) and 2 * inv_freq.shape[0] == rot_dim and dim % 8 == 0 and \
            (dim + rot_dim) % 8 == 0 and tuple(key_up.shape) == (num_heads, kv_rank, dim) and \
            tuple(q.shape) == (meta.num_tokens, num_heads * (dim + rot_dim)) and padded_dim >= kv_rank + rot_dim
        if not fused:
            return super().latent_queries(self.dense(q), key_up, num_heads, dim, rot_dim, padded_dim, inv_freq, magnitude,
                                          neighbours, meta)
        self._own(source, key_up, inv_freq)
        T = meta.num_tokens
        table = self._rope_table(meta, inv_freq)
        out = self._empty((T, num_heads * padded_dim), torch.bfloat16)
        _check(self._ops.distie_latent_queries(
            source, _code(source), slices, dim + rot_dim, key_up, _code(key_up), out,
            padded_dim, T, num_heads, kv_rank, dim, rot_dim // 2, table, float(magnitude),
            1 if neighbours else 0, self._stream()), "latent_queries")
        return out

    def heads_linear(self, x, weight, in_stride, out_stride, out=None):
        x = self.dense(x)
        self._own(x, weight, out)
        if weight.dim() != 3:
            raise KernelError("heads_linear: the weight is [heads, N, K]")
        H, N, K = weight.shape
        T = x.shape[0]
        if x.shape[1] != H * in_stride or K > in_stride or N > out_stride:
            raise KernelError("heads_linear: x is [T, heads * in_stride] with in_stride >= K, out_stride >= N")
        if out is None:
            make = torch.empty if N == out_stride else torch.zeros
            out = make((T, H * out_stride), dtype=x.dtype, device=self.device)
        elif out.dtype != x.dtype or tuple(out.shape) != (T, H * out_stride):
            raise KernelError("heads_linear: out is [T, heads * out_stride] of x's dtype")
        _check(self._ops.distie_heads_linear(x, _code(x), in_stride, weight, _code(weight),
                                             out, out_stride, T, H, N, K, self._stream()), "heads_linear")
        return out

    def rope_heads(self, x, in_stride, in_offset, out, out_stride, out_offset, num_heads, inv_freq, magnitude,
                   neighbours, meta):
        x = self.dense(x)
        self._own(x, out, inv_freq)
        T = x.shape[0]
        if x.dtype != out.dtype or x.shape[1] != num_heads * in_stride or tuple(out.shape) != (T, num_heads * out_stride) \
                or T != meta.num_tokens:
            raise KernelError("rope_heads: x [T, heads * in_stride] and out [T, heads * out_stride] of one dtype")
        table = self._rope_table(meta, inv_freq)
        _check(self._ops.distie_rope_heads(x, _code(x), in_stride, in_offset, out, out_stride,
                                           out_offset, T, num_heads, inv_freq.shape[0], table,
                                           float(magnitude), 1 if neighbours else 0, self._stream()), "rope_heads")
        return out

    def glu_mul(self, gate_up, kind):
        if kind == "silu":
            return self.silu_mul(gate_up)
        if kind not in self.ACTIVATIONS:
            raise KernelError(f"glu_mul: no activation named {kind!r}")
        return self._glu_mul(gate_up, self.ACTIVATIONS[kind])

    def clamped_glu(self, gate_up, limit, slope, up_shift):
        if not limit > 0:
            raise KernelError("clamped_glu: the limit must be positive")
        return self._glu_mul(gate_up, len(self.ACTIVATIONS), (float(limit), float(slope), float(up_shift)))

    def _glu_mul(self, gate_up, kind, clamp=(0.0, 1.0, 0.0)):
        if isinstance(gate_up, (PendingNorm, PendingProduct)):
            gate_up = self.dense(gate_up)
        slices, source, dtype = 1, gate_up, gate_up.dtype
        if isinstance(gate_up, PartialSums):
            slices, source = gate_up.slices, gate_up.data
        self._own(source)
        rows, two = gate_up.shape
        out = self._empty((rows, two // 2), dtype)
        _check(self._ops.distie_glu_mul(source, _code(source), slices, out, _code(out), rows,
                                        two // 2, kind, *clamp, self._stream()), "glu_mul")
        return out

    def silu_mul(self, gate_up):
        if isinstance(gate_up, (PendingNorm, PendingProduct)):
            gate_up = self.dense(gate_up)
        slices, source, dtype = 1, gate_up, gate_up.dtype
        if isinstance(gate_up, PartialSums):
            slices, source = gate_up.slices, gate_up.data
        self._own(source)
        rows, two = gate_up.shape
        out = self._empty((rows, two // 2), dtype)
        _check(self._ops.distie_silu_mul(source, _code(source), slices, out, _code(out),
                                         rows, two // 2, self._stream()), "silu_mul")
        return out

    def gather_rows(self, x, rows):
        x = self.dense(x)
        self._own(x, rows)
        out = self._empty((rows.shape[0], x.shape[1]), x.dtype)
        _check(self._ops.distie_gather_rows(x, rows, out, rows.shape[0],
                                            x.shape[1] * x.element_size(), x.shape[0], self._stream()), "gather_rows")
        return out

    def argmax(self, logits):
        self._own(logits)
        if logits.dtype != torch.float32:
            raise KernelError("argmax reads float32 logits")
        rows, vocab = logits.shape
        out = self._empty(rows, torch.int32)
        parts = self._ops.distie_argmax_parts(rows, vocab)
        values = indexes = None
        if parts > 1:
            values = self._empty(rows * parts, torch.float32)
            indexes = self._empty(rows * parts, torch.int32)
        _check(self._ops.distie_argmax(logits, out, rows, vocab,
                                       values if parts > 1 else None,
                                       indexes if parts > 1 else None, self._stream()), "argmax")
        return out

    def sample(self, logits, temperature, seeds, counters):
        self._own(logits, temperature, seeds, counters)
        if logits.dtype != torch.float32 or temperature.dtype != torch.float32 or \
                seeds.dtype != torch.int64 or counters.dtype != torch.int64:
            raise KernelError("sample: logits/temperature float32, seeds/counters int64")
        rows, vocab = logits.shape
        out = self._empty(rows, torch.int32)
        parts = self._ops.distie_argmax_parts(rows, vocab)
        values = indexes = sums = None
        if parts > 1:
            values = self._empty(rows * parts, torch.float32)
            indexes = self._empty(rows * parts, torch.int32)
            sums = self._empty(rows * parts, torch.float32)
        _check(self._ops.distie_sample(logits, temperature, seeds,
                                       counters, out, rows, vocab,
                                       values if parts > 1 else None,
                                       indexes if parts > 1 else None,
                                       sums if parts > 1 else None, self._stream()), "sample")
        return out
