"""Linears of few rows by tiles of 32 and of 64 rows: the bits of the kernel that streams weights, either side of the step between them."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# (one row, a tile of 32 and one row beside it; outputs of part of a tile, K of one step and of fewer than there are stages)
@pytest.mark.parametrize("m", [9, 31, 32, 33])
@pytest.mark.parametrize("n, ks", [(8, (64, 64)), (68, (128, 64)), (130, (64, 448)), (4100, (320, 64)), (2560, (2560, 10240))])
def test_tiles_of_32_rows(m, n, ks):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + n + sum(ks))
    rows = [torch.randn(m, k, generator=gen).bfloat16().to(DEV) for k in ks]
    weights = [torch.randn(n, k, generator=gen).bfloat16().to(DEV) for k in ks]
    results = []
    try:
        for mode in (1, 2):
            fast.set_skinny_wide(mode)
            out = torch.zeros(m + 1, n, device=DEV)
            out[m] = 7.0
            assert fast.linear_pair_accumulate(rows[0], weights[0], None, rows[1], weights[1], None, out[:m])
            assert bool((out[m] == 7.0).all())
            results.append(out[:m].clone())
    finally:
        fast.set_skinny_wide(1)
    assert torch.equal(*results)
    want = sum(a.double() @ w.double().T for a, w in zip(rows, weights))
    assert float((results[0].double() - want).norm() / want.norm()) < 2.0 ** -20
