"""A step of single tokens of the decaying matrix memory, its token shift and its projections, against float64."""

from __future__ import annotations

import pytest
import torch

from tests.plain import bokorax_plain as plain

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("heads, d, rank", [(3, 16, 5), (2, 20, 64), (1, 4, 1), (32, 64, 64), (5, 100, 300), (2, 128, 512)])
def test_single_tokens_in_one_launch(heads, d, rank, dtype):
    """Rows of requests in any slots beside rows without one, several steps, decays from 1 to 0. The bounds: fp32 sums of up to 512 terms in
    other orders; in bf16 the output's rounding (2^-9) and the hardware's exponential."""
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(heads + d + rank)
    width, dim, eps, slots = heads * d, 28, 1e-6, [2, -1, 0, 3]
    n = len(slots)
    state = torch.randn(5, width * d + dim, generator=gen).to(DEV)
    kept = {s: state[s, :width * d].double().cpu().view(heads, d, d) for s in slots if s >= 0}
    before = state.clone()
    w2 = (torch.randn(width, rank, generator=gen) * 2 * rank ** -0.5).to(dtype)
    w0, u, gain = torch.randn(width, generator=gen) * 2, torch.randn(width, generator=gen), 1 + 0.2 * torch.randn(width, generator=gen)
    for step in range(3):
        rkvg = torch.randn(n, 4 * width + 8, generator=gen).to(dtype)
        low, x = torch.tanh(torch.randn(n, rank, generator=gen)).to(dtype), torch.randn(n, dim, generator=gen)
        out = torch.full((n, width + 4), float("nan"), dtype=dtype, device=DEV)[:, :width]
        on = rkvg.to(DEV)
        parts = [on[:, i * width:(i + 1) * width] for i in range(4)]
        assert core.decayed_step(*parts, low.to(DEV), w2.to(DEV), w0.to(DEV), u.to(DEV), gain.to(DEV), state, x.to(DEV),
                                 torch.tensor(slots, dtype=torch.int32, device=DEV), out, heads, d, eps)
        decay = torch.exp(-torch.exp(low.double() @ w2.double().T + w0.double())).view(n, heads, d)
        r, k, v, g = (rkvg[:, i * width:(i + 1) * width].double().view(n, heads, d) for i in range(4))
        for row, slot in enumerate(slots):
            if slot < 0:
                assert not bool(out[row].any())
                continue
            kv = k[row][:, :, None] * v[row][:, None, :]
            o = ((kept[slot] + u.double().view(heads, d, 1) * kv) * r[row][:, :, None]).sum(dim=1)
            kept[slot] = decay[row][:, :, None] * kept[slot] + kv
            want = plain.rms(o, eps) * gain.double().view(heads, d) * g[row]
            off = (out[row].double().cpu().view(heads, d) - want).norm(dim=1) / want.norm(dim=1)
            assert float(off.max()) <= (2.0 ** -16 if dtype == torch.float32 else 2.0 ** -8)
            here = state[slot, :width * d].double().cpu().view(heads, d, d)
            assert float((here - kept[slot]).norm() / kept[slot].norm()) <= (2.0 ** -20 if dtype == torch.float32 else 2.0 ** -17)
            assert torch.equal(state[slot, width * d:].cpu(), x[row])
    for spare in (1, 4):
        assert torch.equal(state[spare], before[spare])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("dim, counts", [(4, [1]), (1028, [3, 1, 2]), (2048, [1] * 9), (2048, [2047, 5, 1, 2049]), (6000, [1400])])
def test_token_shift_four_channels_at_a_time(dim, counts, dtype):
    """Rows that start and that go on from a kept row, tokens that fill a thread's four and that do not. One product and sum a
    number in fp32, then the type's rounding."""
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(dim + len(counts))
    n, slots = sum(counts), [(-1 if i == 1 else i) for i in range(len(counts))]
    x, kept, mu = torch.randn(n, dim, generator=gen), torch.randn(len(counts) + 1, dim + 8, generator=gen), torch.rand(5, dim, generator=gen)
    cu = torch.tensor([0] + counts).cumsum(0)
    as_int = lambda v: torch.as_tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    out = torch.full((5, n, dim), float("nan"), dtype=dtype, device=DEV)
    core.token_shift(x.to(DEV), kept.to(DEV)[:, 8:], mu.to(DEV), as_int(torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))), as_int(cu),
                     as_int(slots), out)
    before = torch.cat([x[:1], x[:-1]])
    for r, slot in enumerate(slots):
        before[cu[r]] = kept[slot, 8:] if slot >= 0 else 0.0
    want = x.double() + (before.double() - x.double()) * mu.double()[:, None]
    tol = 2.0 ** -22 if dtype == torch.float32 else 2.0 ** -8
    assert bool(((out.double().cpu() - want).abs() <= tol * (x.double().abs() + before.double().abs())).all())


@pytest.mark.parametrize("n", [1, 8, 15, 16, 17, 32])
@pytest.mark.parametrize("k, sizes", [(8, [3]), (72, [16, 50, 1]), (2048, [2048, 2048, 2048, 2048, 64]), (1032, [40] * 8)])
def test_several_linears_in_one_launch(n, k, sizes):
    """Sums of bf16 products in fp32, an activation, one rounding to bf16 (2^-9 of a number; sums that cancel: of their terms)."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(n + k)
    inputs = torch.randn(len(sizes), n, k, generator=gen).bfloat16()
    weights = [(torch.randn(s, k, generator=gen) * k ** -0.5).bfloat16() for s in sizes]
    acts = [(0, 3, 5, 0, 2)[i % 5] for i in range(len(sizes))]
    wide = torch.full((n, sum(sizes) + 6), 7.0, dtype=torch.bfloat16, device=DEV)
    at = [sum(sizes[:i]) for i in range(len(sizes))]
    outs = [wide[:, a:a + s] for a, s in zip(at, sizes)]
    assert fast.linears_few_bf16(list(inputs.to(DEV)), [w.to(DEV) for w in weights], outs, acts)
    for i, (a, w, act) in enumerate(zip(inputs, weights, acts)):
        full = a.double() @ w.double().T
        want = {0: full, 2: full.clamp(min=0.0), 3: full * torch.sigmoid(full), 5: torch.tanh(full)}[act]
        slack = 2.0 ** -8 * want.abs() + 2.0 ** -16 * (a.double().abs() @ w.double().abs().T) + 1e-6
        assert bool(((outs[i].double().cpu() - want).abs() <= slack).all())
    assert bool((wide[:, sum(sizes):] == 7.0).all())
