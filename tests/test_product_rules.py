"""Which kernel a product or a step's attention goes to: the rules alone, without a GPU. Each line names a call on one side of a
boundary where the kernels of both sides were measured."""

import ctypes

import numpy as np
import pytest
import torch

from distie_amd.csrc import build
from distie_amd.kernels.hip_ops import HipOps
from distie_amd.kernels.interface import BatchMeta


@pytest.fixture(scope="module")
def rules():
    ops = HipOps.__new__(HipOps)                   # the rules alone: nothing of this touches a device
    ops._ops = ctypes.CDLL(str(build.ensure("ops")))
    ops._declare()
    ops._tile_plans, ops._large_plans, ops._compute_units, ops.library_timed_portion = {}, {}, 256, 0
    return ops


@pytest.mark.parametrize("kind,rows,weight,captured,timed,tiles", [
    # rotation in the epilogue: weights that the kernels of 16 rows take stay with them as far as those go
    ("rotary", 80, (1536, 1024), True, 0, False), ("rotary", 96, (2048, 1536), True, 0, False),
    ("rotary", 160, (1536, 1024), False, 0, True), ("rotary", 79, (1536, 1024), False, 0, False),
    ("rotary", 97, (1536, 1024), True, 0, True),
    ("rotary", 193, (1536, 1024), False, 0, True), ("rotary", 79, (4608, 3584), True, 0, False),
    ("rotary", 80, (4608, 3584), True, 0, True), ("rotary", 512, (2048, 1536), False, 0, True),
    ("rotary", 640, (2048, 1536), True, 0, False), ("rotary", 640, (2048, 1536), False, 0, True),
    ("rotary", 1101, (2048, 1536), True, 0, False), ("rotary", 224, (4608, 3584), False, 0, True),
    ("rotary", 224, (4608, 3584), False, 512, False),
    # gated
    ("gated", 32, (17920, 1536), True, 0, False), ("gated", 33, (17920, 1536), True, 0, True),
    ("gated", 64, (8192, 1024), True, 0, False), ("gated", 88, (8192, 1024), True, 0, True),
    ("gated", 88, (9728, 896), True, 0, False), ("gated", 96, (4096, 512), True, 0, False),
    ("gated", 160, (4096, 512), False, 0, True), ("gated", 224, (4096, 512), False, 0, True),
    ("gated", 224, (16384, 2048), True, 0, False), ("gated", 301, (17920, 1536), False, 0, True),
    ("gated", 320, (17920, 1536), False, 0, False), ("gated", 640, (8192, 1024), True, 0, False),
    ("gated", 899, (8192, 1024), False, 0, True),
    # the reader adds the slices
    ("down", 64, (1536, 8960), True, 0, True), ("down", 64, (3584, 18944), True, 0, False),
    ("down", 72, (3584, 18944), True, 0, False), ("down", 80, (4096, 11008), True, 0, True),
    ("down", 96, (3584, 18944), True, 0, True), ("attn_out", 64, (5120, 5120), True, 0, False),
    ("attn_out", 96, (1024, 1024), True, 0, False), ("attn_out", 97, (1024, 1024), True, 0, True),
    ("attn_out", 97, (1024, 1024), True, 192, False), ("attn_out", 384, (1536, 1536), True, 0, False),
    ("down", 900, (3072, 8192), False, 0, False), ("down", 1024, (1536, 8960), False, 0, True),
    ("down", 1100, (1536, 8960), False, 0, False),
    # portions of a prompt against large weights: as far as they were measured, and where the library was not timed
    ("down", 2048, (3584, 18944), False, 0, True), ("down", 2017, (3584, 18944), False, 512, True),
    ("down", 2049, (3584, 18944), False, 0, False), ("down", 8192, (3584, 18944), False, 0, False),
    ("down", 1600, (5120, 27648), False, 0, True), ("down", 1800, (5120, 27648), False, 0, False),
    ("down", 1400, (4096, 11008), False, 0, False),
    # whole K
    ("attn_out", 1200, (1536, 1536), False, 0, True), ("attn_out", 1400, (1536, 1536), True, 0, False),
    ("qkv", 576, (4352, 1024), True, 0, True), ("qkv", 576, (4352, 1024), True, 576, False),
    ("qkv", 1400, (3072, 768), True, 0, False),
    ("qkv", 1400, (3072, 768), False, 0, True), ("qkv", 2049, (3072, 768), False, 0, False),
])
def test_products_in_tiles(rules, kind, rows, weight, captured, timed, tiles):
    rules.captured, rules.library_timed_rows = captured, timed
    if kind in ("rotary", "gated"):
        plan = rules._tiles(rows, *weight, kind)
    else:
        plan = rules._tiles(rows, *weight, "plain", 0.0 if kind in rules.ADDS_SLICES else rules.SUM_SLICES_US)
    assert (plan is not None) == tiles
    if plan is not None:
        shape, slices = plan
        stages = weight[1] // 64
        assert 0 <= shape <= 4 and -(-stages // -(-stages // slices)) == slices and (kind not in ("rotary", "gated") or slices == 1)


def test_plans_are_kept_apart_by_what_the_rule_reads(rules):
    rules.captured, rules.library_timed_rows = False, 0
    assert rules._tiles(90, 1536, 1024, "rotary") is not None
    rules.captured = True
    assert rules._tiles(90, 1536, 1024, "rotary") is None
    assert rules._tiles(2048, 3584, 18944, "plain", 0.0) is not None
    rules.library_timed_portion = 2040               # classes of 32 rows
    assert [rules._tiles(rows, 3584, 18944, "plain", 0.0) is None for rows in (1400, 2016, 2017, 2048)] == [False, False, True, True]
    rules.library_timed_portion = 0


@pytest.mark.parametrize("kind,rows,weight,takes", [
    # gated: nearly always; small weights from where they fill a few compute units
    ("gated", 64, (37888, 3584), True), ("gated", 80, (37888, 3584), True), ("gated", 80, (17920, 1536), True),
    ("gated", 65, (8192, 1024), False), ("gated", 193, (8192, 1024), True), ("gated", 2048, (17920, 1536), True),
    ("gated", 301, (17920, 1536), True), ("gated", 97, (4096, 512), False), ("gated", 2048, (17912, 1536), False),
    ("gated", 2048, (17920, 1544), False),
    # rotation: beyond one round of the smaller tiles
    ("rotary", 512, (2048, 1536), False), ("rotary", 576, (2048, 1536), True), ("rotary", 301, (3072, 2048), False),
    ("rotary", 352, (3072, 2048), True), ("rotary", 640, (1536, 1024), False), ("rotary", 704, (1536, 1024), True),
    ("rotary", 256, (4608, 3584), False), ("rotary", 1792, (4608, 3584), True), ("rotary", 2048, (4608, 3584), True),
    ("rotary", 2048, (7168, 5120), False), ("rotary", 4096, (2048, 1536), True), ("rotary", 4097, (2048, 1536), False),
    ("rotary", 2304, (4608, 3072), True), ("rotary", 2305, (4608, 3072), False),
    # plain: where the count comes to a rate that neither the smaller tiles nor the library reach
    ("down", 301, (1536, 8960), False), ("down", 2048, (1536, 8960), True), ("down", 128, (3584, 18944), False),
    ("down", 301, (3584, 18944), True), ("down", 2048, (1024, 2048), False), ("attn_out", 1024, (1536, 1536), False),
    ("attn_out", 2048, (1536, 1536), True), ("qkv", 1024, (1024, 1024), False), ("qkv", 640, (8448, 2048), True),
    ("qkv", 2048, (8448, 2048), False), ("attn_out", 4096, (1536, 1536), True), ("attn_out", 4097, (1536, 1536), False),
    ("down", 2304, (2048, 8192), True), ("down", 2305, (2048, 8192), False), ("down", 4096, (1536, 8960), True), ("down", 4097, (1536, 8960), False),
    ("gated", 8192, (17920, 1536), True),
    # few rows
    ("gated", 8, (17920, 1536), False), ("gated", 9, (17920, 1536), True), ("gated", 16, (4096, 512), False),
    ("gated", 17, (4096, 512), True), ("down", 16, (2048, 8192), False), ("down", 17, (2048, 8192), True),
    ("down", 64, (1536, 8960), False), ("attn_out", 64, (2048, 2048), False), ("attn_out", 17, (3584, 3584), True),
    ("head", 16, (151936, 1536), False), ("head", 17, (151936, 1536), True), ("head", 64, (32768, 2048), False),
    ("rotary", 64, (37888, 3584), False), ("qkv", 64, (8448, 2048), False)])
def test_products_in_large_tiles(rules, kind, rows, weight, takes):
    rules.captured, rules.library_timed_rows = False, 0
    cut_us = None if kind in ("rotary", "gated") else 0.0 if kind in rules.ADDS_SLICES else rules.SUM_SLICES_US
    plan = rules._large(rows, *weight, kind if cut_us is None else "plain", (), cut_us)
    assert (plan is not None) == takes


@pytest.mark.parametrize("N,K", [(16, 256), (40, 320), (1536, 8960), (152064, 3584), (4608, 18944)])
def test_large_tiles_plans_are_launches_that_the_kernel_takes(rules, N, K):
    for rows in (1, 32, 33, 64, 65, 128, 129, 777, 2048, 16384):
        for mode in (0, 1, 2):
            for cut_us in (None, 0.0, 4.5):
                shape, slices, us = ctypes.c_int(-1), ctypes.c_int(-1), ctypes.c_float(-1)
                taken = rules._ops.distie_large_tiles_plan(rows, N, K, mode, cut_us is not None, cut_us or 0.0, ctypes.byref(shape),
                                                           ctypes.byref(slices), ctypes.byref(us))
                assert taken == (N % (16 if mode else 8) == 0)
                if taken:
                    stages = K // 64
                    few = rows <= 64 and mode != 2
                    assert (1 if mode == 2 else 0) <= shape.value <= (13 if few else 7) and (us.value > 0) == (not few)
                    assert -(-stages // -(-stages // slices.value)) == slices.value and (slices.value == 1 or (mode == 0 and cut_us is not None))


def test_large_tiles_leave_what_begins_off_16_bytes(rules):
    rules.captured, rules.library_timed_rows = False, 0
    data = torch.empty(64, dtype=torch.bfloat16)
    assert rules._large(2048, 17920, 1536, "gated", (data, None)) is not None
    assert rules._large(2048, 17920, 1536, "gated", (data[1:], None)) is None


@pytest.mark.parametrize("rows,weight,takes", [
    # the reader adds the slices of K: at up to four rows that pays for long weights only
    (1, (1536, 1536), False), (1, (3584, 3584), False), (1, (1536, 8960), False), (2, (1536, 8960), False), (1, (2560, 10240), True),
    (1, (3072, 7680), False), (4, (3072, 7680), True), (1, (5120, 20480), False), (2, (5120, 20480), True), (4, (5120, 5120), False),
    (3, (2048, 8192), False),
    (5, (2048, 2048), False), (8, (1024, 4096), False), (5, (1536, 3840), True), (8, (1536, 8960), True), (4, (1536, 3840), False),
    (9, (1536, 1536), True), (9, (512, 2048), False), (16, (640, 1600), True), (17, (640, 1600), False),
    (24, (640, 1024), False), (25, (640, 1024), True), (32, (512, 1280), False), (17, (768, 768), True), (32, (768, 768), True),
    (24, (512, 2048), False), (12, (640, 64), False)])
def test_plain_float32_products_of_few_rows(rules, rows, weight, takes):
    assert rules._rows_f32_take(rows, *weight) == takes


def grouped(dim, *sizes):
    return HipOps._grouped_plan(attention(dim), *sizes)


def attention(dim):
    lib = ctypes.CDLL(str(build.ensure(f"attn_d{dim}")))
    lib.distie_attention_f32_plan.argtypes = [ctypes.c_int] * 4 + [ctypes.POINTER(ctypes.c_int)] * 2
    return lib


@pytest.mark.parametrize("dim,requests,heads,kv_heads,visible,plan", [
    # (runs, heads a workgroup, waves): short contexts in one run, a head to itself while workgroups are few
    (128, 1, 12, 2, 30, (1, 1, 4)), (128, 1, 12, 2, 256, (1, 1, 4)), (128, 1, 12, 2, 257, (1, 1, 8)), (128, 1, 12, 2, 512, (1, 1, 8)),
    (128, 1, 12, 2, 513, (3, 1, 4)), (128, 3, 40, 8, 1136, (5, 3, 4)), (128, 1, 12, 2, 4000, (16, 1, 4)),
    (64, 8, 8, 2, 500, (1, 1, 8)), (64, 8, 8, 2, 1000, (4, 1, 4)), (64, 37, 14, 2, 2702, (6, 4, 4)), (64, 64, 8, 2, 1000, (1, 2, 8)),
    (64, 12, 16, 16, 1427, (1, 1, 8)), (64, 2, 16, 16, 1427, (6, 1, 4)), (128, 4, 8, 8, 449, (2, 1, 4)), (128, 32, 8, 8, 449, (1, 1, 8)),
    (64, 146, 8, 2, 288, (1, 4, 8)), (128, 16, 28, 4, 2058, (4, 4, 4)), (128, 32, 12, 2, 1400, (4, 3, 4)), (128, 23, 16, 4, 2048, (5, 4, 4)), (64, 23, 16, 4, 2048, (8, 4, 4)), (192, 140, 3, 1, 714, (3, 3, 4)), (256, 4, 8, 4, 256, (1, 1, 4)), (256, 4, 8, 4, 400, (2, 1, 4)),
    (96, 156, 8, 2, 503, (1, 4, 4)), (96, 1, 8, 2, 466, (1, 1, 8)),
    # heads share a workgroup where their workgroups fill the chip, and four waves where they are more than compute units
    (128, 64, 12, 2, 128, (1, 3, 4)), (128, 16, 12, 2, 4000, (8, 3, 4)), (128, 64, 12, 2, 1000, (1, 3, 8)),
    (128, 29, 12, 2, 389, (1, 2, 8)), (128, 32, 8, 8, 1000, (1, 1, 8)), (128, 64, 28, 4, 700, (1, 4, 4)), (64, 127, 16, 4, 128, (1, 4, 4)),
    # more pairs of token and head than it is for, and a step without keys
    (128, 128, 16, 4, 700, (1, 0, 0)), (128, 1, 12, 2, 0, (1, 0, 0)),
])
def test_float32_attention_of_few_pairs(dim, requests, heads, kv_heads, visible, plan):
    assert grouped(dim, requests, heads, kv_heads, visible) == plan


@pytest.mark.parametrize("dim", [32, 64, 96, 128, 192, 256])
@pytest.mark.parametrize("heads,kv_heads", [(1, 1), (7, 1), (12, 2), (8, 8), (28, 4), (40, 8), (5, 1)])
def test_float32_attention_plans_are_in_bounds(dim, heads, kv_heads):
    for requests in (1, 2, 3, 7, 16, 33, 64, 100, 200, 2047):
        for visible in (1, 63, 64, 65, 300, 449, 1153, 5000, 32768):
            runs, per, waves = grouped(dim, requests, heads, kv_heads, visible)
            if requests * heads >= 2048:
                assert (runs, per, waves) == (1, 0, 0)
                continue
            assert 1 <= runs <= 16 and 1 <= per <= min(4, heads // kv_heads) and (waves == 4 or (waves == 8 and (dim in (32, 64, 128) or dim == 96 and per == 1)))
            assert runs * 64 <= max(64, visible)                    # no more runs than chunks of keys


@pytest.mark.parametrize("dim,splits,group,pairs,together", [
    # four while those workgroups have a compute unit each, eight beyond
    (128, 64, 6, 2, 1), (128, 65, 6, 2, 4), (128, 256, 6, 2, 4), (128, 256, 6, 4, 4), (128, 250, 6, 6, 8), (128, 192, 6, 8, 8),
    (128, 125, 7, 8, 4), (128, 129, 7, 8, 8), (64, 256, 8, 1, 4), (64, 192, 4, 8, 8),
    # heads whose sums fill the LDS, and groups that the kernel does not put together
    (128, 192, 16, 8, 4), (256, 192, 8, 8, 4), (128, 256, 17, 2, 1)])
def test_runs_of_keys_put_together(dim, splits, group, pairs, together):
    assert attention(dim).distie_attention_decode_together(splits, group, pairs) == together


@pytest.mark.parametrize("dim,tokens,requests,heads,kv_heads,max_kv,window,columns", [
    # wide heads, few pairs: short contexts and windows stay with the vector kernel
    (256, 1, 1, 8, 1, 24, 0, False), (256, 8, 8, 8, 1, 1000, 0, False), (192, 6, 6, 24, 2, 139, 0, False), (192, 25, 3, 4, 4, 413, 128, False),
    (256, 120, 120, 24, 2, 36, 0, True), (256, 79, 79, 8, 1, 2011, 0, True), (256, 23, 23, 7, 1, 1232, 0, True),
    (192, 56, 8, 28, 4, 63, 0, True),
    # more pairs, where a wave takes a pair alone otherwise
    (64, 259, 259, 16, 8, 13, 0, False), (128, 82, 82, 28, 4, 21, 0, False), (64, 332, 332, 9, 3, 24, 0, False),
    (192, 240, 240, 10, 2, 13, 0, False), (64, 151, 151, 28, 4, 1002, 0, True), (128, 372, 372, 24, 4, 579, 0, True),
    (256, 430, 119, 12, 2, 306, 0, True), (64, 463, 174, 14, 2, 10000, 128, True), (192, 256, 256, 16, 1, 13, 0, True),
    # up to 128 the vector kernel keeps few pairs whatever their contexts
    (128, 8, 8, 12, 2, 4000, 0, False)])
def test_float32_attention_in_columns_where_it_pays(dim, tokens, requests, heads, kv_heads, max_kv, window, columns):
    lib = attention(dim)
    lib.distie_attention_columns_f32_runs.argtypes = [ctypes.c_int] * 5 + [ctypes.c_int64, ctypes.c_int]
    runs = HipOps._columns_runs(lib, tokens, requests, heads, kv_heads, 16, (heads + 2 * kv_heads) * dim, max_kv, window)
    assert (runs > 0) == columns


def test_wide_heads_on_pages_that_only_columns_take():
    lib = attention(256)
    lib.distie_attention_columns_f32_runs.argtypes = [ctypes.c_int] * 5 + [ctypes.c_int64, ctypes.c_int]
    assert HipOps._columns_runs(lib, 1, 1, 8, 1, 16, 2560, 24, 0) == 0
    assert HipOps._columns_runs(lib, 1, 1, 8, 1, 12, 2560, 24, 0) == 1


def large_plan(rules, rows, N, K, kind, cut_us=None):
    shape, slices, us = ctypes.c_int(-1), ctypes.c_int(-1), ctypes.c_float(-1)
    assert rules._ops.distie_large_tiles_plan(rows, N, K, rules.LARGE_KINDS[kind], cut_us is not None, cut_us or 0.0,
                                              ctypes.byref(shape), ctypes.byref(slices), ctypes.byref(us))
    return shape.value, slices.value, us.value


@pytest.mark.parametrize("kind,rows,weight,cut_us,measured", [
    # a few more tiles of 128 x 128 (shape 7) than compute units: us of those and of the tile that is taken instead
    ("gated", 224, (17920, 1536), None, (30.7, 21.5)), ("gated", 400, (9728, 896), None, (17.1, 12.1)),
    ("gated", 301, (11008, 2048), None, (27.0, 22.4)), ("rotary", 1024, (4608, 3584), None, (58.8, 46.8)),
    ("rotary", 1408, (3072, 2048), None, (33.0, 28.3)), ("plain", 900, (4352, 1024), 4.5, (15.8, 14.1))])
def test_units_with_two_workgroups_are_counted_in_full(rules, kind, rows, weight, cut_us, measured):
    shape, slices, us = large_plan(rules, rows, *weight, kind, cut_us)
    assert shape in (4, 5, 6) and slices == 1 and abs(us / measured[1] - 1) < 0.15


@pytest.mark.parametrize("kind,rows,weight,cut_us,shapes,slices,measured", [
    # few rows of large weights: us of the tile taken (a slower floor made all tiles equal and the first was taken: 72, 74.9, 37.1, 52.0)
    ("gated", 65, (37888, 3584), None, (3, 6), 1, 53.7), ("gated", 128, (37888, 3584), None, (3, 6), 1, 60.5),
    ("plain", 128, (4096, 11008), 0.0, (7,), 6, 30.7), ("plain", 160, (3584, 18944), 0.0, (5,), 8, 42.6)])
def test_plans_of_few_rows_go_by_the_rate_that_memory_reaches(rules, kind, rows, weight, cut_us, shapes, slices, measured):
    shape, cut, us = large_plan(rules, rows, *weight, kind, cut_us)
    assert shape in shapes and cut == slices and abs(us / measured - 1) < 0.15


@pytest.mark.parametrize("rows", [9, 64, 65, 66, 72, 73, 80])
@pytest.mark.parametrize("weight", [(17920, 1536), (16384, 2048), (37888, 3584)])
def test_gated_products_in_large_tiles_leave_no_rows_out(rules, rows, weight):
    """Both sides of the row count where the smaller tiles end: us in these tiles / what there was, 65 rows 17 / 22, 21.5 / 22 and 52 / 72."""
    rules.captured, rules.library_timed_rows = False, 0
    assert rules._large(rows, *weight, "gated", ()) is not None


def test_products_met_before_take_one_look(rules, monkeypatch):
    """A step that is launched kernel by kernel asks for every product of every layer: what was found is kept, by what the rules
    read, and an input off 16 bytes has the other kernels each time."""
    rules.captured, rules.library_timed_rows = False, 0
    data, xs = torch.empty(64, dtype=torch.bfloat16), torch.empty(2, 8, 64, dtype=torch.bfloat16)
    asked = [(M, N, K, kind, cut_us) for M in (9, 32, 64, 301, 2048) for N, K in ((17920, 1536), (1536, 8960), (2048, 1536))
             for kind, cut_us in (("gated", None), ("rotary", None), ("plain", 0.0), ("plain", rules.SUM_SLICES_US))]
    first = [rules._tiled(*a[:4], (data, None), a[4]) for a in asked]
    each = [rules._large_each(rows, 4096, 1024, xs) for rows in (33, 300)]
    for (plan, large), (M, N, K, kind, cut_us) in zip(first, asked):
        assert plan == (rules._large(M, N, K, kind, (), cut_us) or rules._tiles(M, N, K, kind, cut_us))
        assert large == (rules._large(M, N, K, kind, (), cut_us) is not None)
    off = [rules._tiled(*a[:4], (data[1:], None), a[4]) for a in asked]
    assert off == [(rules._tiles(*a), False) for a in asked]
    assert rules._tiled(8, 17920, 1536, "gated", (data,)) == (None, False)
    monkeypatch.setattr(rules, "_ops", None)                 # no rule is walked through again
    assert [rules._tiled(*a[:4], (data, None), a[4]) for a in asked] == first
    assert [rules._large_each(rows, 4096, 1024, xs) for rows in (33, 300)] == each
    assert len(rules._large_plans) <= rules.TILE_PLANS


@pytest.mark.parametrize("kind,rows,weight,takes", [
    # one row of tiles on half of the compute units or fewer, K long: us in these tiles / what there was
    ("gated", 88, (13824, 2560), False),           # 27.2 / 24.7
    ("gated", 128, (16384, 3072), False),          # 33.7 / 32.2
    ("gated", 192, (16384, 3072), False),          # 40.8 / 35.1
    ("gated", 200, (16384, 3072), True),           # 32.5 / 42.6: two rows of them
    ("gated", 88, (20480, 2560), True),            # 29.5 / 34.6: 160 of them
    ("gated", 128, (8192, 1536), False),           # 18.0 / 13.2: 64 of them
    ("gated", 144, (12288, 1536), True),           # 16.7 / 22.0: K short
    ("qkv", 128, (13056, 3072), False),            # 33.0 / 29.0
    ("qkv", 192, (15232, 3584), False),            # 45.4 / 34.9
    ("qkv", 256, (15232, 3584), True),             # 40.0 / 48.5
    ("down", 128, (5120, 20480), True)])           # K cut: 74 / 76
def test_large_tiles_that_would_leave_units_idle(rules, kind, rows, weight, takes):
    rules.captured, rules.library_timed_rows = False, 0
    cut_us = None if kind == "gated" else 0.0 if kind in rules.ADDS_SLICES else rules.SUM_SLICES_US
    assert (rules._large(rows, *weight, "gated" if kind == "gated" else "plain", (), cut_us) is not None) == takes


@pytest.mark.parametrize("gated,rows,weight,through_lds", [
    # gated: us through LDS / on registers
    (True, 8, (8192, 4096), False), (True, 32, (8192, 4096), False),          # 48 / 30, 63 / 49: 171 workgroups of three waves
    (True, 8, (4096, 8192), False), (True, 16, (12288, 3072), False),         # 87 / 33, 41 / 40
    (True, 8, (16384, 2048), False), (True, 12, (16384, 2048), True),         # 33.0 / 31.3, 33.0 / 34.3
    (True, 8, (17920, 1536), True), (True, 7, (17920, 1536), False),          # 27.7 / 28.6
    (True, 8, (24576, 1024), False), (True, 16, (24576, 1024), True),         # 27.3 / 25.4, 27.0 / 28.2
    (True, 1, (37888, 3584), True), (True, 8, (65536, 1536), False),          # 100 / 124
    # plain
    (False, 8, (4096, 4096), False), (False, 16, (4096, 4096), True),         # 24.0 / 22.3, 23.6 / 23.9
    (False, 8, (4096, 11008), False), (False, 17, (4096, 11008), True),       # 50 / 45, 47 / 54
    (False, 8, (3584, 3584), True), (False, 8, (5120, 5120), True),           # 18.8 / 21.7, 28 / 34
    (False, 1, (1536, 8960), True), (False, 33, (1536, 8960), False)])
def test_float32_products_through_lds(rules, gated, rows, weight, through_lds):
    assert (rules._ops.distie_rows_f32_waves(rows, *weight, int(gated)) > 0) == through_lds


@pytest.mark.parametrize("rows,weight,takes", [
    # us in large tiles / what there was
    (256, (6528, 1536), False), (301, (6528, 1536), False), (416, (6528, 1536), True),           # 17.5 / 13.6, 15.8 / 13.4, 16.3 / 16.7
    (192, (8704, 2048), False), (256, (8704, 2048), True),                                       # 20.4 / 17.6, 21.8 / 26.8
    (352, (5440, 1280), False), (416, (5440, 1280), True),                                       # 15.5 / 14.2, 14.3 / 14.8
    (160, (10880, 2560), False), (176, (10880, 2560), True),                                     # 25.3 / 22.9, 24.4 / 38.6
    (480, (4352, 1024), True), (720, (3264, 768), True)])                                        # 11.0 / 12.1, 9.1 / 10.7
def test_wide_weights_in_large_tiles(rules, rows, weight, takes):
    rules.captured, rules.library_timed_rows = False, 0
    assert (rules._large(rows, *weight, "plain", (), rules.SUM_SLICES_US) is not None) == takes


@pytest.mark.parametrize("rows,weight,takes", [
    # us in large tiles / what there was
    (352, (4096, 3072), False), (512, (4096, 3072), False), (576, (4096, 3072), True),           # 31.9 / 24.8, 33.3 / 28.9, 31.2 / 33.3
    (512, (3328, 2560), False), (640, (3328, 2560), True),                                       # 30.4 / 26.6, 30.3 / 31.2
    (416, (4608, 3584), False), (800, (4608, 3584), True),                                       # 35.0 / 31.7, 37.8 / 44.5
    (576, (2048, 1536), True), (416, (3072, 2048), True)])                                       # 17.0 / 17.8, 20 / 20
def test_long_rotating_products_in_large_tiles(rules, rows, weight, takes):
    rules.captured, rules.library_timed_rows = False, 0
    assert (rules._large(rows, *weight, "rotary", ()) is not None) == takes


@pytest.mark.parametrize("rows,weight,takes", [
    # us in large tiles / what there was
    (9, (7168, 1280), False), (16, (7168, 1280), False), (17, (7168, 1280), True),               # 7.6 / 7.2, 7.7 / 7.5, 7.8 / 8.2
    (12, (8192, 1024), False), (17, (8192, 1024), True),                                         # 7.2 / 6.9, 7.1 / 7.5
    (9, (8192, 1536), True), (9, (10240, 1280), True)])                                          # 8.4 / 8.6, 8.3 / 9.7
def test_small_gated_weights_in_large_tiles(rules, rows, weight, takes):
    rules.captured, rules.library_timed_rows = True, 0
    assert (rules._large(rows, *weight, "gated", ()) is not None) == takes


def prompts_plan(heads, portions, single_keys, window=0, known=True, cls=HipOps, kv_heads=None, block_size=16):
    """How a step's portions (tokens, keys behind them) go beside requests that decode behind `single_keys` keys: 28 heads on 4 kv
    heads, 12 on 2."""
    ops = cls.__new__(cls)
    ops.device = torch.device("cpu")
    tokens = [n for n, _ in portions] + [1] * len(single_keys)
    past = [behind for _, behind in portions] + [keys - 1 for keys in single_keys]
    cu_q = np.concatenate([[0], np.cumsum(tokens)]).astype(np.int32)
    meta = BatchMeta(num_tokens=sum(tokens), num_requests=len(tokens), positions=None, token_request=None, cu_q=None, kv_len=None,
                     state_slots=None, max_q=max(tokens), max_kv=max(n + p for n, p in zip(tokens, past)), block_size=block_size,
                     host_cu_q=cu_q if known else None, host_past=np.array(past) if known else None,
                     singles_bound=None if known else len(tokens))
    plan = ops._attention_plan(attention(128), meta, sum(tokens), heads, kv_heads or (heads // 6 if heads == 12 else 4), 128, window)
    return plan["waves"], plan.get("parts")


@pytest.mark.parametrize("heads,portions,window,waves", [
    (12, [(300, 0)], 0, 4), (12, [(300, 900)], 0, 8), (12, [(40, 0), (7, 30)], 0, 2), (12, [(600, 3500)], 0, 8),
    (12, [(600, 5000)], 0, 0), (12, [(300, 2000)], 512, 4), (28, [(667, 0)] * 3, 0, 0), (28, [(667, 0), (667, 0), (600, 1400)], 0, 2),
    (28, [(120, 0)], 0, 4)])
def test_what_requests_decode_behind_is_nothing_to_the_portions_beside_them(heads, portions, window, waves):
    plans = {prompts_plan(heads, portions, [keys, 100], window) for keys in (10, 500, 1100, 2000, 5000, 20000, 100000)}
    assert len(plans) == 1 and plans.pop()[0] == waves


def test_portions_of_a_captured_step_may_have_as_many_keys_as_any_request():
    assert prompts_plan(12, [(300, 0)], [1000], known=False)[0] > 0
    assert prompts_plan(12, [(300, 0)], [20000], known=False)[0] == 0


def test_a_steps_plan_of_attention_is_kept_by_every_rule_that_it_is_made_by():
    read = set()

    class Watched(HipOps):
        def __getattribute__(self, name):
            if name.isupper():
                read.add(name)
            return super().__getattribute__(name)

    for heads in (12, 28):
        for portions in ([(300, 0)], [(64, 4000)], [(667, 0)] * 3, [(600, 5000)], [(1500, 1400)]):
            for known in (True, False):
                prompts_plan(heads, portions, [700], known=known, cls=Watched)
    assert len(read) > 6 and read <= set(HipOps.ATTENTION_PLAN_RULES)


@pytest.mark.parametrize("kv_heads,block_size,takes", [
    (2, 16, True), (1, 65536, True), (255, 65536, True), (256, 65536, False), (4096, 4096, False), (4095, 4096, True), (1 << 20, 16, False),
    (2, 65552, False), (2, 24, False)])
def test_pages_whose_bytes_the_portions_kernel_cannot_count(kv_heads, block_size, takes):
    """It counts a page's bytes in 32 bits: larger pages stay with the tiled kernel."""
    assert bool(attention(128).distie_attention_prefill_keys_fits(kv_heads, block_size)) == takes
    if kv_heads <= 256:                                # (more heads are too many workgroups for so few keys)
        assert (prompts_plan(kv_heads, [(40, 0)], [], kv_heads=kv_heads, block_size=block_size)[0] > 0) == takes
