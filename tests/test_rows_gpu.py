"""Kernels that hold a row, or a head's part of one, at once: sizes around what a thread, a round of loads and a group of slices hold,
against 64 bits."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
F = torch.float64
ROUND = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8}


@pytest.fixture(scope="module")
def ops():
    from distie_amd.kernels.hip_ops import HipOps

    return HipOps(torch.device("cuda:0"))


def rnd(*shape, seed, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).cuda()


def sums(slices, rows, width, seed):
    """-> (what a product leaves, the sum): partial sums, or with one slice the row itself"""
    from distie_amd.kernels.hip_ops import PartialSums

    part = rnd(slices, rows, width, seed=seed)
    return (part[0] if slices == 1 else PartialSums(part, torch.float32)), part.to(F).sum(0)


def rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F)


def near(got, want, slices, dtype, norms):
    """A row's error over its norm: a rounding a slice, eight a norm (its square, sum over lanes, quotient, root and two products; a sum of n
    squares over threads and lanes of at most 40 steps counts its roundings' square root, 6, and half of it), one of the result."""
    bound = (slices + 16 * norms + 4) * 2.0 ** -24 + ROUND[dtype]
    assert got.dtype == dtype
    assert ((got.to(F) - want).norm(dim=-1) <= bound * want.norm(dim=-1)).all()


@pytest.mark.parametrize("width", [4, 252, 260, 1020, 1028, 1536, 2048, 4092, 4100, 8192, 8196, 250])
@pytest.mark.parametrize("slices", [1, 2, 4, 5, 8, 9, 17])
def test_a_chain_of_norms_over_one_row(ops, width, slices):
    """One and two terms, a norm behind and in front, with and without a residual: one and two runs of four columns a thread, a row of its
    last thread alone, rows beyond the registers, and a width that is no multiple of four."""
    rows, eps = 3, 1e-5
    w = [1 + rnd(width, seed=s, scale=0.1) for s in range(4)]
    for terms in (1, 2):
        for normed, post, residual, pre, dtype in ((True, True, True, True, torch.bfloat16), (True, False, False, False, None),
                                                   (False, True, True, True, torch.float32), (False, False, True, False, torch.bfloat16)):
            if terms == 2 and not normed:
                continue
            held = [sums(slices if t == 0 else 3, rows, width, seed=10 + t) for t in range(terms)]
            res = rnd(rows, width, seed=20, scale=2.0) if residual else None
            y = held[0][1]
            if normed:
                y = 0.5 * sum(rms(h[1], w[t], eps) for t, h in enumerate(held))
            if post:
                y = rms(y, w[2], eps)
            before = res.to(F) if residual else None
            got = ops._norm_chain([h[0] for h in held], w[:terms] if normed else None, eps, 0.5, (w[2], eps) if post else None, res,
                                  (w[3], eps) if pre else None, dtype)
            if not residual:
                near(got, y, slices, torch.float32, 1)
                continue
            x = before + y
            near(res, x, slices, torch.float32, normed + post)
            near(got, rms(x, w[3], eps) if pre else x, slices, dtype, 3)


@pytest.mark.parametrize("T", [1, 17, 32, 33, 65])
@pytest.mark.parametrize("dim,rot_dim,kv_rank", [(8, 8, 8), (24, 8, 33), (64, 16, 128), (72, 8, 100), (184, 8, 129), (192, 64, 64),
                                                 (200, 8, 40), (392, 24, 31)])
@pytest.mark.parametrize("slices", [1, 2, 4, 5, 9])
def test_queries_of_a_latent(ops, T, dim, rot_dim, kv_rank, slices):
    """The queries' product with its tail, from a row or its partial sums: ends of a round of columns (64 and 192), of tiles of rows and
    of weight rows. The summed input is rounded to bfloat16 first, as a kernel in front would leave it; then a result is off by its own
    rounding and by 2^-24 of the products' sizes for each of K / 8 steps."""
    from distie_amd.kernels.hip_ops import PartialSums

    heads, padded, width = 3, kv_rank + rot_dim + 5, dim + rot_dim
    part = rnd(slices, T, heads * width, seed=1)
    total = part[0].clone()
    for s in range(1, slices):
        total += part[s]
    q = total.bfloat16()
    up = rnd(heads, kv_rank, dim, seed=2, scale=0.3).bfloat16()
    freq = 10.0 ** -torch.arange(rot_dim // 2, dtype=torch.float32, device="cuda")
    meta = SimpleNamespace(num_tokens=T, positions=torch.arange(T, dtype=torch.int32, device="cuda"))
    ops._rope_table = lambda meta, freq: torch.stack([angle.cos(), angle.sin()], -1).float().contiguous()
    angle = (torch.arange(T, device="cuda").to(F)[:, None] * freq.to(F))
    try:
        got = ops.latent_queries(q if slices == 1 else PartialSums(part, torch.bfloat16), up, heads, dim, rot_dim, padded, freq, 1.0,
                                 False, meta).to(F).view(T, heads, padded)
    finally:
        del ops._rope_table
    x = q.to(F).view(T, heads, width)
    want = torch.stack([x[:, h, :dim].contiguous() @ up[h].to(F).t().contiguous() for h in range(heads)], 1)
    size = torch.stack([x[:, h, :dim].abs().contiguous() @ up[h].to(F).abs().t().contiguous() for h in range(heads)], 1)
    assert ((got[..., :kv_rank] - want).abs() <= 2.0 ** -8 * want.abs() + (dim / 8 + 2) * 2.0 ** -24 * size).all()
    u, v = x[..., dim:dim + rot_dim // 2], x[..., dim + rot_dim // 2:]
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    turned = torch.cat([u * cos - v * sin, v * cos + u * sin], -1)
    most = torch.cat([u.abs() + v.abs()] * 2, -1)
    assert ((got[..., kv_rank:kv_rank + rot_dim] - turned).abs() <= 2.0 ** -8 * turned.abs() + 2.0 ** -21 * most).all()
    assert not got[..., kv_rank + rot_dim:].any()


@pytest.mark.parametrize("q_rank,kv_rank,rot_dim", [(0, 5, 0), (7, 64, 6), (768, 192, 64), (1024, 1028, 8), (1100, 300, 514), (3000, 1200, 64)])
@pytest.mark.parametrize("slices", [1, 3, 4, 5, 9])
def test_norms_of_a_latent(ops, q_rank, kv_rank, rot_dim, slices):
    """The latents' norms and the cache write: rows within a round of loads and beyond it, more pairs than threads."""
    T, P, eps = 3, 16, 1e-5
    down, total = sums(slices, T, q_rank + kv_rank + rot_dim, seed=1)
    q_w = 1 + rnd(q_rank, seed=2, scale=0.1) if q_rank else None
    kv_w = 1 + rnd(kv_rank, seed=3, scale=0.1)
    padded = kv_rank + rot_dim + 3
    k = torch.zeros(2, 1, P, padded, device="cuda")
    v = torch.zeros(2, 1, padded, P, device="cuda")
    slots = torch.tensor([1, 17, 30], dtype=torch.int32, device="cuda")
    meta = SimpleNamespace(num_tokens=T, block_size=P, groups=[SimpleNamespace(slots=slots)])
    got = ops.latent_norm_rope_write(down, q_rank, q_w, kv_rank, kv_w, eps, rot_dim, None, 1.0, False, meta, 0, k, v, True, torch.float32)
    if q_rank:
        near(got, rms(total[:, :q_rank], q_w, eps), slices, torch.float32, 1)
    at = slots.long()
    c = rms(total[:, q_rank:q_rank + kv_rank], kv_w, eps)
    near(k[at // P, 0, at % P, :kv_rank], c, slices, torch.float32, 1)
    assert torch.equal(v[at // P, 0, :kv_rank, at % P], k[at // P, 0, at % P, :kv_rank])
    if rot_dim:
        near(k[at // P, 0, at % P, kv_rank:kv_rank + rot_dim], total[:, q_rank + kv_rank:], slices, torch.float32, 0)
    assert not k[at // P, 0, at % P, kv_rank + rot_dim:].any() and not v[:, 0, kv_rank:].any()


@pytest.mark.parametrize("heads,kv_heads,dim", [(12, 2, 128), (3, 1, 96), (8, 8, 64), (4, 2, 256)])
@pytest.mark.parametrize("keys", [1, 3, 16, 63, 64, 65, 130, 700])
def test_float32_decode_attention_at_the_ends_of_its_chunks(ops, heads, kv_heads, dim, keys):
    """One key, a part of a quarter, of a chunk and of a run, behind pages that hold NaN where no key was written. A score is off by
    (dim + 2) / 2 roundings of its products at most; a tenth of that in the root mean square bounds the result's error."""
    lib = ops.attention_library(dim)
    P, T = 16, 2
    lengths = [keys, max(1, keys // 2)]
    pages = -(-keys // P)
    k = torch.full((2 * pages + 1, kv_heads, P, dim), float("nan"), device="cuda")
    v = torch.full((2 * pages + 1, kv_heads, dim, P), float("nan"), device="cuda")
    table = torch.randperm(2 * pages, generator=torch.Generator().manual_seed(1)).view(2, pages).int() + 1
    k[0], v[0] = 0.0, 0.0
    qkv = rnd(T, (heads + 2 * kv_heads) * dim, seed=2)
    want = torch.empty(T, heads, dim, dtype=F, device="cuda")
    for t, n in enumerate(lengths):
        kk, vv = rnd(kv_heads, n, dim, seed=3 + t), rnd(kv_heads, n, dim, seed=5 + t)
        for j in range(n):
            k[table[t, j // P], :, j % P], v[table[t, j // P], :, :, j % P] = kk[:, j], vv[:, j]
        q = qkv[t, :heads * dim].to(F).view(kv_heads, heads // kv_heads, dim)
        weight = torch.softmax(q @ kk.to(F).transpose(1, 2).contiguous() * dim ** -0.5, -1)
        want[t] = (weight @ vv.to(F)).view(heads, dim)
    import ctypes

    per, waves = ctypes.c_int(), ctypes.c_int()
    runs = lib.distie_attention_f32_plan(T, heads, kv_heads, keys, ctypes.byref(per), ctypes.byref(waves))
    assert per.value > 0
    dev = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")  # noqa: E731
    positions, request, table = dev([n - 1 for n in lengths]), dev([0, 1]), table.cuda()
    out = torch.empty(T, heads * dim, device="cuda")
    part_o, part_ml = torch.empty(runs, T, heads, dim, device="cuda"), torch.empty(runs, T, heads, 2, device="cuda")
    assert lib.distie_attention_generic(
        qkv.data_ptr(), 0, qkv.stride(0), k.data_ptr(), v.data_ptr(), 0, positions.data_ptr(), request.data_ptr(), table.data_ptr(), pages,
        None, out.data_ptr(), T, heads, kv_heads, P, dim ** -0.5, 0, None, 0.0, None, part_o.data_ptr(), part_ml.data_ptr(), runs,
        per.value, waves.value, torch.cuda.current_stream().cuda_stream) == 0
    got = out.to(F).view(T, heads, dim)
    assert ((got - want).norm(dim=-1) <= 0.1 * (dim + 2) / 2 * 2.0 ** -24 * want.norm(dim=-1) + 2.0 ** -23 * want.norm(dim=-1)).all()


@pytest.mark.parametrize("heads,kv_heads", [(3, 3), (4, 2), (6, 2), (8, 2)])
@pytest.mark.parametrize("keys", [1, 63, 65, 700])
def test_float32_decode_attention_of_heads_beyond_the_registers(ops, heads, kv_heads, keys):
    """One to four query heads of a size whose keys take several rounds and whose values several parts, the last of them shorter."""
    test_float32_decode_attention_at_the_ends_of_its_chunks(ops, heads, kv_heads, 320, keys)


@pytest.mark.parametrize("T", [5461, 5462, 5500])
@pytest.mark.parametrize("dim,kv_rank", [(72, 129), (200, 129), (192, 64)])
def test_queries_of_a_latent_where_workgroups_are_many(ops, T, dim, kv_rank):
    """Three heads: where the input begins to go through LDS, and where one wave's columns are all there are."""
    test_queries_of_a_latent(ops, T, dim, 8, kv_rank, 1)


def test_queries_of_as_many_heads_as_a_grid_holds(ops):
    """Each head's tail has a workgroup of its own while a grid holds them, here not: the same bits as of a third of the heads."""
    heads, dim, rot_dim, kv_rank, T = 65535, 8, 2, 8, 2
    q, up = rnd(T, heads * (dim + rot_dim), seed=1).bfloat16(), rnd(heads, kv_rank, dim, seed=2).bfloat16()
    freq = torch.ones(1, device="cuda")
    meta = SimpleNamespace(num_tokens=T, positions=torch.arange(T, dtype=torch.int32, device="cuda"), scratch={})
    call = lambda q, up: ops.latent_queries(q.contiguous(), up.contiguous(), len(up), dim, rot_dim, 11, freq, 1.0, False, meta).view(T, -1, 11)  # noqa: E731
    parts = zip(q.view(T, 3, -1).unbind(1), up.view(3, -1, kv_rank, dim).unbind(0))
    assert torch.equal(call(q, up), torch.cat([call(*p) for p in parts], 1))
