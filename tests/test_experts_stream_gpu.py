"""The experts' linears of few pairs where weights and pairs go straight into LDS (K in steps of 64, up to eight pairs of an expert at a time), at its edges."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# K: one step for one of the four waves, less than a step each, as many steps as stages and more, the loop for any K; N: less than 16 rows, a rest
@pytest.mark.parametrize("n, k", [(8, 64), (24, 128), (36, 192), (40, 704), (1408, 2048), (20, 832), (40, 200)])
# pairs per expert: one and eight (the stream), nine to sixteen (16 columns by the loop), seventeen (32 by the loop), thirty-three and forty (32 by the loop, the
# rest of up to eight by the stream)
@pytest.mark.parametrize("counts", [(1, 0, 3), (8, 9, 1), (16, 17, 2), (33, 0, 40)])
@pytest.mark.parametrize("per", [1, 3])
def test_one_linear_of_listed_pairs(per, counts, n, k):
    """fp32 outputs against float64: a sum of K products is off by at most (K + 4) 2^-24 of their magnitudes. Rows of pairs that chose nobody stay."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(n + k + per)
    owners = torch.tensor([e for e, c in enumerate(counts) for _ in range(c)] + [len(counts)] * 2)        # (the last choose no expert with weights)
    chosen = owners[torch.randperm(owners.numel(), generator=gen)].int()
    pairs = chosen.numel()
    a = torch.randn(-(-pairs // per), k, generator=gen).bfloat16()
    w = (torch.randn(len(counts), n, k, generator=gen) * k ** -0.5).bfloat16()
    out = torch.full((pairs, n), 7.0, device=DEV)
    ad, wd, cd = a.to(DEV), w.to(DEV), chosen.to(DEV)
    fast._check(fast.lib().ka_experts_few_bf16(ad.data_ptr(), k, per, wd.data_ptr(), cd.data_ptr(), pairs, len(counts), n, k, 0, 0, 0.0, 0.0, 0.0,
                                               out.data_ptr(), n, 1, fast.stream_ptr()))
    out = out.cpu().double()
    for p, e in enumerate(chosen.tolist()):
        if e == len(counts):
            assert bool((out[p] == 7.0).all())
            continue
        x = a[p // per].double()
        assert bool(((out[p] - w[e].double() @ x).abs() <= (k + 4) * 2.0 ** -24 * (w[e].double().abs() @ x.abs())).all()), p


@pytest.mark.parametrize("k", [192, 2048])
def test_a_pair_has_the_same_bits_alone_and_among_others(k):
    """Alone and among eight pairs of its expert (the stream), nine and sixteen (the loop of 16), thirty-three (the loop of 32, the last one by the stream)."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(k)
    a, w = torch.randn(33, k, generator=gen).bfloat16().to(DEV), torch.randn(1, 72, k, generator=gen).bfloat16().to(DEV)
    outs = {}
    for pairs in (1, 8, 9, 16, 33):
        chosen, outs[pairs] = torch.zeros(pairs, dtype=torch.int32, device=DEV), torch.empty(pairs, 72, device=DEV)
        fast._check(fast.lib().ka_experts_few_bf16(a.data_ptr(), k, 1, w.data_ptr(), chosen.data_ptr(), pairs, 1, 72, k, 0, 0, 0.0, 0.0, 0.0,
                                                   outs[pairs].data_ptr(), 72, 1, fast.stream_ptr()))
    for pairs, out in outs.items():
        assert torch.equal(out, outs[33][:pairs]), pairs
