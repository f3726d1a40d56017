"""The experts' linears listed by expert at the edges of their tiles, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("gated, clamped", [(True, False), (True, True), (False, False)], ids=["silu", "clamped", "plain"])
@pytest.mark.parametrize("n, dim, ff, n_experts, top, tile", [
    (1, 64, 64, 1, 1, 64), (130, 128, 64, 9, 3, 64), (203, 192, 320, 5, 1, 64), (96, 64, 128, 3, 2, 128), (1030, 256, 192, 30, 4, 128),
    (1, 64, 64, 2, 1, 256), (400, 64, 448, 4, 2, 256), (513, 128, 64, 4, 1, 256), (1100, 192, 128, 2, 1, 256)])
def test_listed_experts_in_tiles(n, dim, ff, n_experts, top, tile, gated, clamped):
    """One list row, tiles that end before their last row and columns that end inside a tile, K from one step of 64 on, experts
    that nobody chose, identity experts among the choices (their pairs stay as they are). The bound: a hidden number is
    rounded once to bf16 (2^-9 of it) and the products sum in fp32; the 2-norm of a pair's outputs is then off by about
    2^-9 of itself, twice that is allowed."""
    from kestrel_amd.engine.batch import Workspace
    from kestrel_amd.ops import fast
    from kestrel_amd.ops.linear import ACT_GATED, activation_code, pair_rows
    from kestrel_amd.parts.specs import GateClamp

    gen = torch.Generator().manual_seed(n + dim + ff)
    rows = 2 * ff if gated else ff
    act = activation_code("silu") | ACT_GATED if gated else activation_code("relu_squared")
    chosen_tile = fast.lib().ka_experts_gemm_tile(n * top, n_experts, rows, dim, act, dim)
    assert chosen_tile == (64 if n * top * 5 <= n_experts * 256 else 128)       # (256 takes more tiles than the chip has CUs)
    h = torch.randn(n, dim, generator=gen).bfloat16()
    gate, up = ((torch.randn(n_experts, ff, dim, generator=gen) * dim ** -0.5).bfloat16() for _ in range(2))
    down = (torch.randn(n_experts, dim, ff, generator=gen) * ff ** -0.5).bfloat16()
    outputs = n_experts + (2 if n % 2 else 0)                  # (odd numbers of tokens: with two identity experts)
    chosen = torch.stack([torch.randperm(outputs, generator=gen)[:top] for _ in range(n)]).to(torch.int32)
    if n_experts > 4:
        chosen[chosen == 3] = n_experts - 1                    # nobody's expert, and one with more rows than the others
    first = torch.stack([pair_rows(gate[e], up[e]) for e in range(n_experts)]) if gated else up
    y = torch.full((n * top, dim), 7.0, device=DEV)
    clamp = GateClamp(0.7, 1.702, 1.0) if clamped else None
    assert fast.lib().ka_experts_gemm_tile(12288, 62, 1792 if gated else 896, 4096, act, 4096) == 256
    assert fast.experts_feed_forward_bf16(h.to(DEV), first.to(DEV), down.to(DEV), chosen.to(DEV), None, y, act, Workspace(torch.device(DEV)), clamp=clamp,
                                          tile=tile)
    want = torch.full((n * top, dim), 7.0, dtype=torch.float64)
    flat = chosen.view(-1).long()
    x = h.double().repeat_interleave(top, 0)
    for e in range(n_experts):
        at = (flat == e).nonzero()[:, 0]
        g, u = x[at] @ gate[e].double().T, x[at] @ up[e].double().T
        if clamped:
            g, u = g.clamp(max=0.7), u.clamp(-0.7, 0.7)
            hidden = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        else:
            hidden = g * torch.sigmoid(g) * u if gated else u.clamp(min=0.0) ** 2
        want[at] = hidden @ down[e].double().T
    off = (y.cpu().double() - want).norm(dim=1) / want.norm(dim=1).clamp(min=1e-3)
    assert bool((off[flat < n_experts] <= 2.0 ** -8).all())
    assert bool((y.cpu()[flat >= n_experts] == 7.0).all())
