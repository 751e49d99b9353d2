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
