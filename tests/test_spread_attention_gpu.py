"""Paged attention in 32 bits where keys come in whole lines: edges of its chunks, its forms by waves and head size, its options."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def plain(q, keys, values, lo, hi, places, scale, o):
    """One token, one head in 64 bits: ``keys [n, hd]``, ``values [n, hdv]``."""
    kept = min(o.get("keep_first", 0), lo)
    at = torch.tensor([j for j in range(keys.shape[0]) if j < kept or lo <= j < hi], dtype=torch.long)
    s = (keys[at] @ q) * scale
    if o.get("softcap"):
        s = o["softcap"] * torch.tanh(s / o["softcap"])
    if o.get("slope") is not None:
        s = s - o["slope"] * (places - at)
    if o.get("bias") is not None:
        s = s + o["bias"][(places - at).clamp(0, len(o["bias"]) - 1)]
    if o.get("sink") is not None:
        s = torch.cat([s, o["sink"].view(1)])
    p = torch.softmax(s, 0)[:len(at)] if s.numel() else s
    return p @ values[at]


# (of 32 heads 3 and 16 tokens: four waves a token on 256 CUs, 17 and 150: one)
@pytest.mark.parametrize("n", [3, 16, 17, 150])
@pytest.mark.parametrize("heads, kv_heads, maps, hd, hdv, page", [(32, 32, 1, 64, 64, 16), (32, 8, 1, 80, 80, 16), (32, 4, 1, 4, 20, 4), (32, 2, 1, 256, 132, 12),
                                                                (32, 4, 2, 36, 256, 32), (32, 8, 1, 128, 96, 64), (32, 1, 1, 16, 8, 128)])
@pytest.mark.parametrize("options", ["", "window sink", "window kept slopes gate", "bias softcap head_gate sinks"])
def test_spread_attention(n, heads, kv_heads, maps, hd, hdv, page, options):
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(n + hd + hdv + len(options))
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    n_rows, longest = 3, 291
    pages = -(-longest // page)
    order = torch.randperm(n_rows * pages, generator=gen).to(torch.int32).view(n_rows, pages)
    # every place without a key holds what is no number
    keys, values = rnd(n_rows, longest, kv_heads, hd), rnd(n_rows, longest, kv_heads // maps, hdv)
    k_cache = torch.full((n_rows * pages, kv_heads, page, hd), float("nan"))
    v_cache = torch.full((n_rows * pages, kv_heads // maps, hdv, page), float("nan"))
    for r in range(n_rows):
        for j in range(longest):
            k_cache[order[r, j // page], :, j % page] = keys[r, j]
            v_cache[order[r, j // page], :, :, j % page] = values[r, j]
    his = [1, 2, 3, 4, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 290, longest]
    hi = torch.tensor([his[(i * 7 + n) % len(his)] for i in range(n)], dtype=torch.int32)
    row = torch.arange(n, dtype=torch.int32) % n_rows
    lo = (hi - 1 - torch.arange(n, dtype=torch.int32) * 13 % 70).clamp(min=0) if "window" in options else None
    if lo is not None and n > 3:
        lo[1] = hi[1]                                          # (no key at all)
    qkv = rnd(n, heads * hd + 4)
    q = qkv[:, 4:]
    extra, per_head = {}, [{} for _ in range(heads)]
    if "window sink" in options:
        extra["sink"] = 0.3
        per_head = [dict(o, sink=torch.tensor(0.3, dtype=torch.float64)) for o in per_head]
    if "sinks" in options:
        sinks = rnd(heads)
        extra["sinks"] = sinks.to(DEV)
        per_head = [dict(o, sink=sinks[h].double()) for h, o in enumerate(per_head)]
    if "kept" in options:
        extra["keep_first"] = 5
        per_head = [dict(o, keep_first=5) for o in per_head]
    if "slopes" in options:
        slopes = rnd(heads).abs() * 0.05
        extra["slopes"] = slopes.to(DEV)
        per_head = [dict(o, slope=slopes[h].double()) for h, o in enumerate(per_head)]
    if "bias" in options:
        bias = rnd(heads, 50)
        extra["bias_table"] = bias.to(DEV)
        per_head = [dict(o, bias=bias[h].double()) for h, o in enumerate(per_head)]
    if "softcap" in options:
        extra["softcap"] = 2.0
        per_head = [dict(o, softcap=2.0) for o in per_head]
    gate = None
    if "gate" in options:
        by_head = "head_gate" in options
        gate = rnd(n, heads if by_head else heads * hdv)
        extra.update(gate=gate.to(DEV), gate_per_head=by_head)
    places = hi - 1
    scale = hd ** -0.5
    out = torch.full((n, heads * hdv), float("nan"), device=DEV)
    core.attention_generic(qkv.to(DEV)[:, 4:], k_cache.to(DEV), v_cache.to(DEV), order.to(DEV), row.to(DEV), lo.to(DEV) if lo is not None else None, hi.to(DEV), out,
                           scale, heads, kv_heads, hd, value_dim=hdv, positions=places.to(DEV), maps=maps, **extra)
    want = torch.zeros(n, heads, hdv, dtype=torch.float64)
    for t in range(0, n, max(1, n // 12)):
        for h in range(0, heads, 5):
            vh = h // maps // (heads // kv_heads)
            kvh = vh * maps + h % maps
            want[t, h] = plain(q[t, h * hd:(h + 1) * hd].double(), keys[row[t], :, kvh].double(), values[row[t], :, vh].double(),
                               int(lo[t]) if lo is not None else 0, int(hi[t]), int(places[t]), scale, per_head[h])
            if gate is not None:
                want[t, h] *= torch.sigmoid(gate[t, h].double() if "head_gate" in options else gate.view(n, heads, hdv)[t, h].double())
    got = out.cpu().double().view(n, heads, hdv)
    assert torch.isfinite(got).all()
    got, want = got[::max(1, n // 12), ::5], want[::max(1, n // 12), ::5]
    # scores of fp32 operands (a few units of 2^-24 times some 8), their exponentials and averages
    assert float((got - want).abs().max()) <= 2.0 ** -18 * max(1.0, float(want.abs().max()))
    assert float((got - want).norm() / want.norm()) < 2.0 ** -20


# (chunks of 64, 32 and 16 keys: some hold nothing but keys that the table shuts out; tokens in four waves and in one)
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("n", [3, 40])
def test_keys_that_a_table_shuts_out(hd, n):
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(n + hd)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    heads, page, longest = 32, 16, 200
    pages = -(-longest // page)
    keys, values, q = rnd(longest, heads, hd), rnd(longest, heads, hd), rnd(n, heads * hd)
    whole = torch.zeros(2, pages * page, heads, hd)
    whole[0, :longest], whole[1, :longest] = keys, values
    k_cache = whole[0].view(pages, page, heads, hd).transpose(1, 2).contiguous()
    v_cache = whole[1].view(pages, page, heads, hd).permute(0, 2, 3, 1).contiguous()
    hi = torch.tensor([(60, 17, 200)[t % 3] for t in range(n)], dtype=torch.int32)
    # distances below 20 count for the first heads, those of 20 and more for the others (a row of 17 keys then sees none)
    bias = rnd(heads, 21)
    bias[:16, 20] = float("-inf")
    bias[16:, :20] = float("-inf")
    out = torch.full((n, heads * hd), float("nan"), device=DEV)
    core.attention_generic(q.to(DEV), k_cache.to(DEV), v_cache.to(DEV), torch.arange(pages, dtype=torch.int32, device=DEV).view(1, pages),
                           torch.zeros(n, dtype=torch.int32, device=DEV), None, hi.to(DEV), out, hd ** -0.5, heads, heads, hd,
                           positions=(hi - 1).to(DEV), bias_table=bias.to(DEV))
    for t in range(n):
        for h in (0, 15, 16, 31):
            seen = [j for j in range(int(hi[t])) if (int(hi[t]) - 1 - j < 20) == (h < 16)]
            want = torch.zeros(hd, dtype=torch.float64)
            if seen:
                s = keys[seen, h].double() @ q[t, h * hd:(h + 1) * hd].double() * hd ** -0.5
                s = s + bias[h].double()[(int(hi[t]) - 1 - torch.tensor(seen)).clamp(max=20)]
                want = torch.softmax(s, 0) @ values[seen, h].double()
            got = out[t, h * hd:(h + 1) * hd].cpu().double()
            assert float((got - want).abs().max()) <= 2.0 ** -18 * max(1.0, float(want.abs().max())), (t, h)
