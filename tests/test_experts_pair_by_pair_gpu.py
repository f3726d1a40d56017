"""The experts' linears pair by pair: rows fetched ahead have the bits of the plain loop, at the edges of its forms."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("k", [512, 520, 704, 1024, 1032, 2040, 2048, 2056, 4088, 4096, 4104])
@pytest.mark.parametrize("n_out, gated, f32", [(1, True, False), (37, True, False), (64, False, True), (30, False, False)])
def test_rows_ahead_have_the_bits_of_the_loop(k, n_out, gated, f32):
    from kestrel_amd.ops import core
    from kestrel_amd.ops.linear import ACT_GATED, activation_code

    gen = torch.Generator().manual_seed(k + n_out)
    experts, tokens, top = 3, 4, 2
    a = torch.randn(tokens, k, generator=gen).bfloat16()
    w = (torch.randn(experts, n_out * (2 if gated else 1), k, generator=gen) * k ** -0.5).bfloat16()
    chosen = torch.tensor([0, 2, 1, 3, 2, 0, 4, 1], dtype=torch.int32)       # (3 and 4: no experts with weights)
    act = activation_code("silu") | (ACT_GATED if gated else 0)
    wide = torch.zeros(tokens, k + 1, dtype=torch.bfloat16)                  # (rows that no piece of eight fits: the loop)
    wide[:, :k] = a
    results = []
    for rows in (a.to(DEV), wide.to(DEV)[:, :k]):
        out = torch.full((tokens * top, n_out), 5.0, dtype=torch.float32 if f32 else torch.bfloat16, device=DEV)
        core.experts_linear(rows, top, w.to(DEV), chosen.to(DEV), out, act)
        results.append(out.cpu())
    assert torch.equal(*results)
    for p, e in enumerate(chosen.tolist()):
        if e >= experts:
            assert bool((results[0][p] == 5.0).all())
            continue
        z = a[p // top].double() @ w[e].double().T
        want = torch.nn.functional.silu(z[0::2]) * z[1::2] if gated else torch.nn.functional.silu(z)
        # fp32 sums; a bf16 result is rounded once (2^-9)
        assert float((results[0][p].double() - want).abs().max()) <= (2.0 ** -18 if f32 else 2.0 ** -8) * max(1.0, float(want.abs().max()))
