"""The decaying matrix memory by chunks, against the recurrence in float64."""

from __future__ import annotations

import pytest
import torch

from tests.plain import bokorax_plain as plain

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("decays", ["slow", "mixed", "sudden"])
@pytest.mark.parametrize("heads, d", [(3, 16), (2, 48), (4, 64), (2, 128), (1, 224)])
def test_decaying_memory_by_chunks(heads, d, decays):
    """Rows fed in pieces that begin and end anywhere in a chunk and in a block of it, a row without a request, pieces of one
    token through the other kernel in between (the state is one and the same). "sudden": decays from 1 to exactly 0 beside
    each other. The bound: the output is rounded to bf16 (2^-9); what fp32 sums are off is far less, unless the terms cancel, as
    they may in a few of some thousand tokens (2^-6 for any one of them, 2^-8.5 over all; the state at a finer bound in
    test_decayed_walks_gpu.py)."""
    from kestrel_amd.ops import core, fast

    gen = torch.Generator().manual_seed(heads * 1000 + d)
    width, dim, eps = heads * d, 24, 1e-6
    pieces = [[64, 1, 100], [1, 17, 3], [130, 1, 63], [40, 0, 16], [5, 33, 1]]
    slots = [2, 0, 3, -1, 1]
    state = torch.zeros(5, width * d + dim, device=DEV)
    u, gain = torch.randn(width, generator=gen), 1 + 0.2 * torch.randn(width, generator=gen)
    data, got = [], [[] for _ in pieces]
    for p in pieces:
        n = sum(p)
        rkvg = torch.randn(n, 4 * width, generator=gen).bfloat16()
        pre = torch.randn(n, width, generator=gen)
        if decays == "slow":
            pre = pre - 5.0
        elif decays == "sudden":
            pre = torch.where(pre > 1.0, 30.0, torch.where(pre < 0.0, -40.0, pre * 4.0 - 2.0))
            pre[:, 0] = float("inf")                           # a channel that never keeps anything
        data.append((rkvg, pre))
    as_int = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    at = [0] * len(pieces)
    for step in range(3):
        live = [r for r, p in enumerate(pieces) if p[step] > 0]
        cut = [slice(at[r], at[r] + pieces[r][step]) for r in live]
        rkvg = torch.cat([data[r][0][c] for r, c in zip(live, cut)]).to(DEV)
        pre = torch.cat([data[r][1][c] for r, c in zip(live, cut)]).to(DEV).contiguous()
        n = rkvg.shape[0]
        cu = [0]
        for c in cut:
            cu.append(cu[-1] + c.stop - c.start)
        out = torch.full((n, width), float("nan"), dtype=torch.bfloat16, device=DEV)
        x = torch.randn(n, dim, generator=gen).to(DEV)
        parts = [rkvg[:, i * width:(i + 1) * width] for i in range(4)]
        operands = (*parts, pre, u.to(DEV), gain.to(DEV), state, x, as_int(cu), as_int([slots[r] for r in live]), out, heads, d, eps)
        if step == 1:
            core.decayed_memory(*operands)
        else:
            scratch = torch.full((fast.gated_chunks_scratch(n, len(live), heads, d, d),), float("nan"), device=DEV)
            assert fast.decayed_chunks_bf16(*operands, torch.full((n, width), float("nan"), device=DEV), scratch)
        for i, r in enumerate(live):
            got[r].append(out[cu[i]:cu[i + 1]].double().cpu())
            if slots[r] >= 0:
                assert torch.equal(state[slots[r], width * d:], x[cu[i + 1] - 1])
            at[r] += cut[i].stop - cut[i].start
    for r, (rkvg, pre) in enumerate(data):
        here = torch.cat(got[r])
        if slots[r] < 0:
            assert not bool(here.any())
            continue
        q, k, v, g = rkvg.double().split(width, dim=1)
        decay = torch.exp(-torch.exp(pre.double()))
        for a in range(heads):
            c = slice(a * d, (a + 1) * d)
            o, last = plain.wkv_recurrence(q[:, c], k[:, c], v[:, c], decay[:, c], u[c].double())
            want = plain.rms(o, eps) * gain[c].double() * g[:, c]
            off = (here[:, c] - want).norm(dim=1) / want.norm(dim=1)
            assert float(off.max()) <= 2.0 ** -6 and float(off.square().mean().sqrt()) <= 2.0 ** -8.5, (r, a, float(off.max()), float(off.square().mean().sqrt()))
            kept = state[slots[r], a * d * d:(a + 1) * d * d].double().cpu().view(d, d)
            assert float((kept - last).norm() / last.norm()) <= 2.0 ** -12
