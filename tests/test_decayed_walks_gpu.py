"""The decaying matrix memory over prompt portions: as near to 64 bits as the walk over whole rows, whatever the decays are, and causal
whatever the tokens hold."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EPS = 1e-6


def _operands(n, heads, d, seed):
    gen = torch.Generator().manual_seed(seed)
    width = heads * d
    rkvg = torch.randn(n, 4 * width, generator=gen).bfloat16()
    pre = torch.randn(n, width, generator=gen)
    return rkvg, pre, torch.randn(width, generator=gen), 1 + 0.2 * torch.randn(width, generator=gen), torch.randn(2, width * d, generator=gen)


def _run(how, rkvg, pre, u, gain, state, heads, d):
    """Rows 0 and 1 of the step are the requests in slots 1 and 0, the first with a third of the tokens."""
    from kestrel_amd.ops import core, fast

    n, width = rkvg.shape[0], heads * d
    as_int = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    rkvg, state, out = rkvg.to(DEV), state.clone().to(DEV), torch.full((n, width), float("nan"), dtype=torch.bfloat16, device=DEV)
    parts = [rkvg[:, i * width:(i + 1) * width] for i in range(4)]
    operands = (*parts, pre.to(DEV), u.to(DEV), gain.to(DEV), state, None, as_int([0, n // 3, n]), as_int([1, 0]), out, heads, d, EPS)
    if how == "rows":
        core.decayed_memory(*operands)
    else:
        scratch = torch.full((fast.gated_chunks_scratch(n, 2, heads, d, d),), float("nan"), device=DEV)
        assert fast.decayed_chunks_bf16(*operands, torch.full((n, width), float("nan"), device=DEV), scratch)
    return out.cpu(), state.cpu()


@pytest.mark.parametrize("decays", ["slow", "mixed", "dead runs"])
@pytest.mark.parametrize("heads, d", [(2, 16), (3, 64), (1, 80), (2, 128), (1, 224)])
def test_chunks_are_as_near_to_64_bits_as_whole_rows(heads, d, decays):
    """"dead runs": 24 to 40 tokens whose decays are next to nothing, then slow ones, within a chunk and across its end. The bound: per key
    channel a state is a sum of some hundred fp32 products, each decayed token by token; the hardware's exponentials are off by a few
    2^-23 of their argument, for decays near 1 by that of themselves. 2^-16 of the channel's norm, and, over all
    channels, twice what whole rows are off and 2^-22 more (a chunk multiplies its decays first, the state behind)."""
    n = 400
    rkvg, pre, u, gain, state = _operands(n, heads, d, heads * 1000 + d)
    if decays == "slow":
        pre = pre - 5.0
    elif decays == "dead runs":
        pre = pre * 0.5 - 7.0
        for at, length in ((20, 24), (70, 40), (150, 30), (270, 24), (330, 33)):
            pre[at:at + length] = 4.0 + pre[at:at + length].abs() * 0.1        # (decays of e^-60 to e^-120 a token)
    off = {}
    for how in ("rows", "chunks"):
        _out, kept = _run(how, rkvg, pre, u, gain, state, heads, d)
        worst, whole = 0.0, []
        for slot, tokens in ((1, slice(0, n // 3)), (0, slice(n // 3, n))):
            q, k, v, _g = rkvg[tokens].double().split(heads * d, dim=1)
            decay = torch.exp(-torch.exp(pre[tokens].double()))
            for a in range(heads):
                c = slice(a * d, (a + 1) * d)
                S = state[slot, a * d * d:(a + 1) * d * d].double().view(d, d).clone()
                for t in range(k.shape[0]):
                    S = decay[t, c, None] * S + k[t, c, None] * v[t, None, c]
                got = kept[slot, a * d * d:(a + 1) * d * d].double().view(d, d)
                worst = max(worst, float(((got - S).norm(dim=1) / S.norm(dim=1)).max()))
                whole.append((got - S).norm() / S.norm())
        assert worst <= 2.0 ** -16, how
        off[how] = float(torch.stack(whole).square().mean().sqrt())
    assert off["chunks"] <= 2.0 * off["rows"] + 2.0 ** -22


@pytest.mark.parametrize("d", [48, 64, 128])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_what_a_token_holds_does_not_travel_backwards(d, bad):
    """One value, one key and one decay's pre-activation that are no numbers, at places within a block, at its edge and at a chunk's: the tokens
    before, the other request and the other head are the same bits as without."""
    heads, n = 2, 300
    rkvg, pre, u, gain, state = _operands(n, heads, d, d)
    clean, kept = _run("chunks", rkvg, pre, u, gain, state, heads, d)
    assert bool(torch.isfinite(clean.float()).all())
    for at in (107, 115, 100 + 63, 100 + 64, 299):
        for part in (1, 2, 3):
            dirty, dirty_pre = rkvg.clone(), pre.clone()
            if part == 3:
                dirty_pre[at, 5] = float("nan")
            else:
                dirty[at, part * heads * d + 5] = bad
            out, after = _run("chunks", dirty, dirty_pre, u, gain, state, heads, d)
            assert torch.equal(out[:at], clean[:at]) and torch.equal(out[:, d:], clean[:, d:])
            assert torch.equal(after[1], kept[1]) and torch.equal(after[0, d * d:], kept[0, d * d:])
            assert part == 3 or not bool(torch.isfinite(out[at, :d].float()).all())
