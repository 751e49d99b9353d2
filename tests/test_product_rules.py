"""Which kernel a product goes to, by its rows, its weight and what reads its result: the rule alone, without a GPU. Each line
names a product on one side of a boundary where the kernels of both sides were measured."""

import ctypes

import pytest

from distie_amd.csrc import build
from distie_amd.kernels.hip_ops import HipOps


@pytest.fixture(scope="module")
def rules():
    ops = HipOps.__new__(HipOps)                   # the rules alone: nothing of this touches a device
    ops._ops = ctypes.CDLL(str(build.ensure("ops")))
    ops._declare()
    ops._tile_plans, ops._compute_units, ops.library_timed_portion = {}, 256, 0
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
