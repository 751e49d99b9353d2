"""Kernels that walk a step's rows in groups and carry a state a request: requests that begin at every place of a group, single rows beside
portions, and widths that leave lanes of the last wave without a channel, against 64 bits."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
F = torch.float64
HALF, SINGLE = 2.0 ** -8, 2.0 ** -24          # of a result rounded to bfloat16, of one float32 operation


@pytest.fixture(scope="module")
def ops():
    from distie_amd.kernels.hip_ops import HipOps

    return HipOps(torch.device("cuda:0"))


def rnd(*shape, seed, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).cuda()


def step(cuts, block_size=16):
    """A step whose requests bring `cuts` rows each, every one behind a context of its own length, in state rows and pages that do not lie
    in their order -> (meta, pages)"""
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    past = [0 if b == 0 else 7 * b % 19 for b in range(len(cuts))]
    cu, slots, request, positions, pages = [0], [], [], [], 0
    for b, n in enumerate(cuts):
        own = list(range(pages, pages + -(-(past[b] + n) // block_size)))
        pages += len(own)
        own = own[::-1]
        slots += [own[p // block_size] * block_size + p % block_size for p in range(past[b], past[b] + n)]
        request += [b] * n
        positions += range(past[b], past[b] + n)
        cu.append(cu[-1] + n)
    B = len(cuts)
    return SimpleNamespace(num_tokens=cu[-1], num_requests=B, cu_q=i32(cu), host_cu_q=np.asarray(cu), max_q=max(cuts), token_request=i32(request),
                           positions=i32(positions), state_slots=i32([(5 * b + 2) % 31 for b in range(B)]), all_decode=max(cuts) == 1,
                           block_size=block_size, groups=[SimpleNamespace(slots=i32(slots))], scratch={}), pages


def convolved(x, filters, state, meta):
    """-> (results, the sizes of what they are added up from, the state behind the step), in 64 bits"""
    taps = filters.shape[1]
    out, size, behind = [], [], state.to(F)
    for b, (a, e) in enumerate(zip(meta.host_cu_q, meta.host_cu_q[1:])):
        at = (5 * b + 2) % 31
        rows = torch.cat([behind[at], x[a:e].to(F)])
        terms = [rows[j:j + e - a] * filters[:, j].to(F) for j in range(taps)]
        out.append(sum(terms))
        size.append(sum(t.abs() for t in terms))
        behind[at] = rows[-(taps - 1):]
    return torch.cat(out), torch.cat(size), behind


@pytest.mark.parametrize("value_dim", [8, 72, 136, 264])
@pytest.mark.parametrize("taps", [2, 3, 4])
def test_convolved_values_of_requests_that_begin_anywhere_in_a_group(ops, value_dim, taps):
    """q, k and v with filters and head norms: 16 rows of v are one group of lanes' work, and a wave's last channels may be eight. What is
    behind the first request begins at every row of the second group: a portion, or a single row and two portions. A value is off by its
    own rounding and one of each product and sum; what is carried is copied."""
    H, G, D, eps = 3, 2, 72, 1e-5
    E, padded = value_dim, max(D, value_dim)
    channels = H * D + G * (D + E)
    filters = rnd(channels, taps, seed=1, scale=0.5).bfloat16()
    norms = (1 + rnd(D, seed=2, scale=0.2), 1 + rnd(D, seed=3, scale=0.2), eps)
    for begin in range(16):
        for rest in ((40,), (1, 2, 1, 1, 37)):
            meta, pages = step((16 + begin, *rest))
            T = meta.num_tokens
            x, state = rnd(T, channels, seed=4 + begin).bfloat16(), rnd(31, taps - 1, channels, seed=5 + begin, scale=2.0)
            k = torch.zeros(pages, G, 16, padded, dtype=torch.bfloat16, device="cuda")
            v = torch.zeros(pages, G, padded, 16, dtype=torch.bfloat16, device="cuda")
            want, size, behind = convolved(x, filters, state, meta)
            q = ops.conv_rope_kv_write(x, filters, state, meta, 0, k, v, None, 1.0, H, G, D, E, padded, True, True, None, norms)
            at = meta.groups[0].slots.long()
            got = v[at // 16, :, :E, at % 16].to(F).reshape(T, G * E)
            values, sizes = want[:, -G * E:], size[:, -G * E:]
            assert ((got - values).abs() <= HALF * values.abs() + taps * SINGLE * sizes).all(), (begin, rest)
            assert torch.equal(state.to(F), behind), (begin, rest)
            for got, heads, first, weight in ((q.view(T, H, padded), H, 0, norms[0]), (k[at // 16, :, at % 16], G, H * D, norms[1])):
                u = want[:, first:first + heads * D].view(T, heads, D)
                scale = weight.to(F) / torch.sqrt((u * u).mean(-1, keepdim=True) + eps)
                off = (HALF * u.abs() + (taps + 16) * SINGLE * size[:, first:first + heads * D].view(T, heads, D)) * scale.abs()
                assert ((got[..., :D].to(F) - u * scale).norm(dim=-1) <= off.norm(dim=-1)).all(), (begin, rest, heads)
                assert not got[..., D:].any()


def scanned(x, dt, dt_bias, a_log, skip, state, meta, H, P, N, G):
    """-> (outputs, the sizes of what they are added up from, the state behind the step and its sizes, the largest exponent of a decay over a
    chunk of 64 rows), in 64 bits"""
    x, state, sizes, bend = x.to(F), state.to(F), state.to(F).abs(), 0.0
    d = torch.nn.functional.softplus(dt.to(F) + dt_bias.to(F), threshold=80.0)
    a = torch.exp(-torch.exp(a_log.to(F)) * d)
    out, size = torch.empty(len(x), H, P, dtype=F, device="cuda"), torch.empty(len(x), H, P, dtype=F, device="cuda")
    for b in range(meta.num_requests):
        at = (5 * b + 2) % 31
        s, most, first, end = state[at], sizes[at], *meta.host_cu_q[b:b + 2]
        bend = max([bend] + [-a[t:min(t + 64, end)].log().sum(0).min().item() for t in range(first, end, 64)])
        for t in range(first, end):
            v = x[t, :H * P].view(H, 1, P)
            B, C = (x[t, H * P + i * G * N:H * P + (i + 1) * G * N].view(G, N).repeat_interleave(H // G, 0)[:, :, None] for i in (0, 1))
            s = a[t][:, None, None] * s + d[t][:, None, None] * B * v
            most = a[t][:, None, None] * most + d[t][:, None, None] * (B * v).abs()
            out[t] = (s * C).sum(1) + skip.to(F)[:, None] * v[:, 0]
            size[t] = (most * C.abs()).sum(1) + (skip.to(F)[:, None] * v[:, 0]).abs()
        state[at], sizes[at] = s, most
    return out.view(len(x), H * P), size.view(len(x), H * P), state, sizes, bend


def scan_case(ops, cuts, H, P, N, G, dtype):
    """A result is off by a few roundings of each of its terms' products and of their sum over at most 64 rows and N state rows in eights, and
    by those of the two sums of exponents of which a decay's is the difference."""
    meta, _ = step(cuts)
    T = meta.num_tokens
    x, dt = rnd(T, H * P + 2 * G * N, seed=1).to(dtype), rnd(T, H, seed=2).to(dtype)
    bias, a_log, skip = rnd(H, seed=3), rnd(H, seed=4, scale=0.5) - 2, rnd(H, seed=5)
    state = rnd(31, H, N, P, seed=6, scale=2.0)
    want, size, behind, sizes, bend = scanned(x, dt, bias, a_log, skip, state, meta, H, P, N, G)
    got = ops.ssm_scan(x, dt, bias, a_log, skip, state, meta, H, P, N, G)
    assert got.dtype == torch.float32
    for got, want, size in ((got, want, size), (state, behind, sizes)):
        assert ((got.to(F) - want).abs() <= (2 * bend + 64 + N / 8) * SINGLE * size).all()


def test_as_many_heads_as_a_grid_holds(ops):
    """Heads and groups together are more than a grid has rows."""
    scan_case(ops, (33, 1), 65535, 1, 1, 1, torch.float32)


@pytest.mark.parametrize("T", [255, 256, 257, 300])
@pytest.mark.parametrize("channels", [8, 424, 520])
@pytest.mark.parametrize("taps", [2, 3, 4])
def test_convolution_of_two_rows_a_thread(ops, T, channels, taps):
    """From 256 rows on a thread has two, which may belong to one request or to two, one of them a single row; channels that leave lanes of the
    last wave without any. With a bias and silu, whose slope is below 1.1, or with the row itself added."""
    cuts = [1, 2, 3, 1, 1, 5, 1, 2, 61, 1, 1, 3, 2, 1, 4]
    cuts += [T - sum(cuts) - 2, 1, 1]
    filters, bias = rnd(channels, taps, seed=1, scale=0.5).bfloat16(), rnd(channels, seed=2)
    x, first = rnd(T, channels, seed=3).bfloat16(), rnd(31, taps - 1, channels, seed=4, scale=2.0)
    meta, _ = step(cuts)
    sums, size, behind = convolved(x, filters, first, meta)
    for residual, act in ((False, "silu"), (True, None)):
        state = first.clone()
        got = ops.causal_conv(x, filters, state, meta, residual, bias, act)
        want = sums + bias.to(F) + (x.to(F) if residual else 0.0)
        off = (taps + 3) * SINGLE * (size + bias.abs() + (x.abs() if residual else 0.0))
        if act:
            want, off = want * torch.sigmoid(want), 1.1 * off + 8 * SINGLE * want.abs()
        assert ((got.to(F) - want).abs() <= HALF * want.abs() + off).all()
        assert torch.equal(state.to(F), behind)


@pytest.mark.parametrize("cuts", [(33, 1, 1, 40, 1), (1,) * 20 + (64,), (65, 1), (1, 200, 2, 1, 3), (32,), (1, 128)])
@pytest.mark.parametrize("H,P,N,G", [(4, 64, 16, 2), (2, 40, 33, 1), (3, 130, 64, 3), (2, 64, 128, 1), (2, 24, 256, 2), (2, 16, 257, 1)])
def test_single_rows_beside_portions_of_state_spaces(ops, cuts, H, P, N, G):
    """Single rows go row by row, portions in chunks; a state of more rows than the row-by-row kernel keeps goes in chunks with both."""
    scan_case(ops, cuts, H, P, N, G, torch.bfloat16 if N % 2 == 0 else torch.float32)


@pytest.mark.parametrize("cuts", [(16,), (17, 1), (64, 1, 63), (65, 16, 1, 130)])
@pytest.mark.parametrize("heads,dim", [(3, 16), (2, 24), (2, 64), (2, 72), (1, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pad", [0, 1])
def test_time_mixing_at_the_ends_of_its_chunks(ops, cuts, heads, dim, dtype, pad):
    """Whole and partial chunks and runs of sixteen rows, heads that fill their channels and others, rows that four values can be read from and
    others. A sum is off by a few roundings of its terms and by those of the decays' exponents, added up over at most 64 rows; the
    norm carries the head's relative error on."""
    meta, _ = step(cuts)
    T, N, rank, eps = meta.num_tokens, heads * dim, 5, 1e-5
    rows = rnd(T, 4 * N + pad, seed=1).to(dtype)
    r, k, v, gates = (rows[:, i * N:(i + 1) * N] for i in range(4))
    low, up, up_bias = rnd(T, rank, seed=2), rnd(N, rank, seed=3, scale=0.3), rnd(N, seed=4, scale=0.3)
    bonus, weight = rnd(N, seed=5), 1 + rnd(N, seed=6, scale=0.2)
    state = rnd(31, heads, dim, dim, seed=7)
    z = torch.tanh(low.to(F)) @ up.to(F).t().contiguous() + up_bias.to(F)
    rate = torch.exp(z).view(T, heads, dim)
    r_, k_, v_ = (t.to(F).reshape(T, heads, dim) for t in (r, k, v))
    u = bonus.to(F).view(heads, dim, 1)
    out, size = torch.empty(T, heads, dim, dtype=F, device="cuda"), torch.empty(T, heads, dim, dtype=F, device="cuda")
    behind, sizes, bend = state.to(F), state.to(F).abs(), 0.0
    for b in range(meta.num_requests):
        at, first, end = (5 * b + 2) % 31, *meta.host_cu_q[b:b + 2]
        bend = max([bend] + [rate[t:min(t + 64, end)].sum(0).max().item() for t in range(first, end, 64)])
        s, most = behind[at], sizes[at]
        for t in range(first, end):
            pair, decay = k_[t][:, :, None] * v_[t][:, None, :], torch.exp(-rate[t])[:, :, None]
            out[t] = ((s + u * pair) * r_[t][:, :, None]).sum(1)
            size[t] = ((most + (u * pair).abs()) * r_[t].abs()[:, :, None]).sum(1)
            s, most = decay * s + pair, decay * most + pair.abs()
        behind[at], sizes[at] = s, most
    g = gates.to(F).view(T, heads, dim)
    normed = out / torch.sqrt((out * out).mean(-1, keepdim=True) + eps)
    factor = weight.to(F).view(heads, dim) * g * torch.sigmoid(g)
    got = ops.wkv_mix(r, k, v, gates, low, up, up_bias, bonus, state, meta, heads, dim, weight, eps, dtype).to(F).view(T, heads, dim)
    # (the decay's logit: rank + 2 roundings of its terms and those of tanh; a decay's relative error is its exponent's absolute one)
    coefficient = (bend * (rank + 8) + 64 + dim / 4) * SINGLE
    off = 2 * coefficient * size.norm(dim=-1) / out.norm(dim=-1) * (normed.norm(dim=-1) * factor.abs().amax(-1))
    want = normed * factor
    assert ((got - want).norm(dim=-1) <= off + ((HALF if dtype == torch.bfloat16 else 0.0) + 16 * SINGLE) * want.norm(dim=-1)).all()
    assert ((state.to(F) - behind).abs() <= coefficient * sizes).all()
