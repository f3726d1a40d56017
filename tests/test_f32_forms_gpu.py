"""32-bit linears at row counts and tile counts where another form of a kernel begins, against float64 and against each other."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# rows: the forms of the weight stream (1, 2, 3, 4, up to 6, 8, 16); columns: two a wave, one (up to 4,096), four (from 8,192 at five rows)
@pytest.mark.parametrize("m", [2, 3, 5, 6, 7, 8])
@pytest.mark.parametrize("n, k", [(130, 2052), (5000, 1024), (8193, 260)])
def test_rows_of_a_weight_stream(m, n, k):
    """Bound: a sum of K products is off by at most (K + 4) 2^-24 of the sum of their magnitudes. A row's bits do not depend on the others'."""
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(m + n + k)
    a, w, bias = torch.randn(m, k, generator=gen).to(DEV), torch.randn(n, k, generator=gen).to(DEV), torch.randn(n, generator=gen).to(DEV)
    out, alone = torch.full((m, n), float("nan"), device=DEV), torch.empty(1, n, device=DEV)
    core.linear_generic(a, w, bias, out)
    want = a.double() @ w.double().T + bias.double()
    assert bool(((out.double() - want).abs() <= (k + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs())).all())
    for r in range(m):
        core.linear_generic(a[r:r + 1], w, bias, alone)
        assert torch.equal(alone[0], out[r])


# tiles of 64 x 32: as many as CUs (steps of 32), one more (steps of 16); of 64 x 64; of 32 x 32; K of one step of 32, of parts cut short
@pytest.mark.parametrize("k", [32, 96, 160, 1056])
@pytest.mark.parametrize("m, n", [(128, 4096), (128, 4160), (250, 4100), (303, 6144), (303, 2048), (33, 8200)])
def test_tiles_and_steps(m, n, k):
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=gen).to(DEV), torch.randn(n, k, generator=gen).to(DEV)
    out, few = torch.full((m, n), float("nan"), device=DEV), torch.empty(17, n, device=DEV)
    core.linear_generic(a, w, None, out)
    assert bool(((out.double() - a.double() @ w.double().T).abs() <= (k + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)).all())
    core.linear_generic(a[:17], w, None, few)
    assert torch.equal(few, out[:17])
