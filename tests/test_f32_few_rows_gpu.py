"""A block's step in 32 bits: two linears a launch and attention with its rotation and cache write, to the bit what the launches one by one give (which other tests hold against 64 bits)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# rows: every form; K: one step, a unit and parts of one, both numbers of fours a thread and the first sizes beyond the smaller; outputs: odd ones, fewer than waves, more
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("k, n1, n2", [(256, 1, 7), (1024, 33, 1024), (1280, 3840, 2561), (2048, 6144, 8192), (2304, 5, 9), (2560, 77, 5120), (2816, 9, 5), (3072, 4, 4)])
@pytest.mark.parametrize("norm", [None, True, False])
def test_two_first_linears(m, k, n1, n2, norm):
    from kestrel_amd.ops import core
    from kestrel_amd.ops.linear import linear

    gen = torch.Generator().manual_seed(m + k)
    rnd = lambda *s: torch.randn(*s, generator=gen).to(DEV)  # noqa: E731
    x, wa, wb = (rnd(m, k) if norm is not None else rnd(m, k + 8)[:, :k]), rnd(n1, k + 4)[:, :k], rnd(n2, k)
    ba, gamma, beta = rnd(n1), rnd(k), rnd(k) if norm else None
    outs = [torch.full((m, n + 3), 7.0, device=DEV) for n in (n1, n2)]
    took = core.linears_first_f32(x, None if norm is None else (gamma, beta, 1e-5), wa, ba, outs[0][:, :n1], 0, wb, None, outs[1][:, :n2], 1)
    assert took == (m * k <= 16384 and (m <= 6 or k <= 2048))      # (seven and eight rows: two fours a thread)
    if not took:
        assert all(bool((o == 7.0).all()) for o in outs)
        return
    h = x
    if norm is not None:
        h = torch.empty_like(x)
        core.layernorm(x, gamma, beta, 1e-5, h)
    want = [torch.empty(m, n, device=DEV) for n in (n1, n2)]
    linear(h, wa, ba, want[0])
    linear(h, wb, None, want[1], act=1)
    assert all(torch.equal(o[:, :n], w) and bool((o[:, n:] == 7.0).all()) for o, n, w in zip(outs, (n1, n2), want))


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("n, k1, k2", [(1, 256, 256), (2047, 2048, 8192), (130, 1024, 1280), (2560, 2560, 10240), (6, 768, 4096)])
def test_two_last_linears(m, n, k1, k2):
    from kestrel_amd.ops import core
    from kestrel_amd.ops.linear import linear

    gen = torch.Generator().manual_seed(m + n)
    rnd = lambda *s: torch.randn(*s, generator=gen).to(DEV)  # noqa: E731
    a1, a2, w1, w2 = rnd(m, k1 + 4)[:, :k1], rnd(m, k2), rnd(n, k1), rnd(n, k2 + 8)[:, :k2]
    b1, rows = rnd(n), rnd(m, n + 5)
    out, want = rows.clone(), rows.clone()
    assert core.linears_last_f32(a1, w1, b1, a2, w2, None, out[:, :n])
    linear(a1, w1, b1, want[:, :n], accumulate=True)
    linear(a2, w2, None, want[:, :n], accumulate=True)
    assert torch.equal(out, want)


def test_what_is_not_covered():
    from kestrel_amd.ops import core

    z = lambda *s, t=torch.float32: torch.zeros(*s, dtype=t, device=DEV)  # noqa: E731
    first = lambda x, wa, wb, act=0: core.linears_first_f32(x, None, wa, None, z(x.shape[0], wa.shape[0]), act, wb, None, z(x.shape[0], wb.shape[0]), 0)  # noqa: E731
    assert first(z(8, 256), z(4, 256), z(4, 256))
    for x, wa, wb in ((z(9, 256), z(4, 256), z(4, 256)), (z(2, 260), z(4, 260), z(4, 260)), (z(2, 256), z(4, 257)[:, 1:], z(4, 256)), (z(2, 3328), z(4, 3328), z(4, 3328)),
                      (z(2, 256), z(4, 256, t=torch.bfloat16), z(4, 256)), (z(1, 256).expand(2, 256), z(4, 256), z(4, 256))):
        assert not first(x, wa, wb)
    last = lambda m, k: core.linears_last_f32(z(m, k), z(4, k), None, z(m, 256), z(4, 256), None, z(m, 4))  # noqa: E731
    assert last(8, 512) and not last(9, 512) and not last(2, 320)


# the token's own key at every place of a chunk and of a page; a row of the batch without a request (slot -1); keys kept from a window's start on
@pytest.mark.parametrize("heads, kv_heads, hd, page, rot, pairing", [(32, 32, 64, 16, 32, "halves"), (32, 8, 80, 16, 32, "halves"), (8, 1, 4, 4, 2, "interleaved"), (6, 2, 128, 64, 128, "interleaved"),
                                                                     (4, 4, 132, 12, 66, "halves"), (2, 1, 256, 128, 256, "halves"), (32, 4, 36, 32, 0, "halves")])
@pytest.mark.parametrize("window", [False, True])
def test_attention_of_single_tokens(heads, kv_heads, hd, page, rot, pairing, window):
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(hd)
    n, longest = 16, 291
    pages = -(-longest // page)
    table = torch.randn(longest, rot, generator=gen).to(DEV) if rot else None
    order = torch.randperm(n * pages, generator=gen).to(torch.int32).view(n, pages)
    caches = [torch.randn(n * pages, kv_heads, *s, generator=gen).to(DEV) for s in ((page, hd), (hd, page))]
    qkv = torch.randn(n, (heads + 2 * kv_heads) * hd + 4, generator=gen).to(DEV)[:, :(heads + 2 * kv_heads) * hd]
    at = torch.tensor([0, 1, 2, 3, 14, 15, 16, 62, 63, 64, 127, 128, 254, 255, 256, 290], dtype=torch.int32)
    slots = torch.tensor([order[i, p // page] * page + p % page for i, p in enumerate(at.tolist())], dtype=torch.int32)
    for i, s in enumerate(slots.tolist()):                       # (nothing that is a number where the token's own key and value go)
        caches[0][s // page, :, s % page] = caches[1][s // page, :, :, s % page] = float("nan")
    slots[4] = -1
    caches[0][order[4, 14 // page], :, 14 % page] = caches[1][order[4, 14 // page], :, :, 14 % page] = 1.0
    lo = (at - torch.arange(n, dtype=torch.int32) * 13 % 70).clamp(min=0).to(DEV) if window else None
    slots, hi, at, order, row = slots.to(DEV), (at + 1).to(DEV), at.to(DEV), order.to(DEV), torch.arange(n, dtype=torch.int32, device=DEV)
    fused, step_by_step, rows, rotated = [c.clone() for c in caches], [c.clone() for c in caches], qkv.clone(), qkv.clone()
    got, want = (torch.full((n, heads * hd), 7.0, device=DEV) for _ in range(2))
    for part in (slice(0, 8), slice(8, 16)):                     # (a workgroup for every CU at the most)
        assert core.attention_step_f32(rows[part], at[part], slots[part], table, *fused, order, row[part], None if lo is None else lo[part], hi[part], got[part], 0.3,
                                       heads, kv_heads, hd, pairing)
    core.rope_cache(rotated, at, slots, table, *step_by_step, heads, kv_heads, hd, page, pairing)
    core.attention_generic(rotated, *step_by_step, order, row, lo, hi, want, 0.3, heads, kv_heads, hd)
    assert torch.equal(rows, qkv) and torch.equal(got, want)
    assert all(torch.equal(a, b) for a, b in zip(fused, step_by_step))
    many = qkv[:1].expand(600, -1).contiguous()                 # (more than that: a launch each)
    big = torch.zeros(600, dtype=torch.int32, device=DEV)
    assert not core.attention_step_f32(many, big, big - 1, table, *fused, order, big, None, big + 1, torch.empty(600, heads * hd, device=DEV), 0.3, heads, kv_heads, hd, pairing)
