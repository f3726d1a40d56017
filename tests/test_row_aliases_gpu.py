"""The launch that ends routed experts and finishes a row of the stream, where its input is the stream itself."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# (the general form; one piece a thread of 256, 512 and 1,024 threads; two of 1,024; several pieces a thread of many rows)
@pytest.mark.parametrize("n, dim", [(3, 102), (3, 1024), (5, 2048), (2, 4096), (3, 8192), (1100, 2048)])
def test_experts_input_may_be_the_stream(n, dim):
    """Identity experts add the row that is about to be written: the same bits as with a copy of it."""
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(n + dim)
    top, E = 4, 3
    rnd = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)  # noqa: E731
    y, x, shared, gain, gain2 = rnd(n * top, dim), rnd(n, dim), rnd(n, dim), rnd(dim), rnd(dim)
    chosen, weights = torch.randint(0, E + 3, (n, top), generator=gen).to(torch.int32).to(DEV), rnd(n, top).abs()
    results = []
    for copied in (False, True):
        stream, rows = x.clone(), torch.full((n, dim), float("nan"), device=DEV)
        core.experts_combine_normed(y, stream.clone() if copied else stream, chosen, weights, E, shared, None, stream, (gain, 1e-5), (gain2, 1e-5), rows)
        results.append((stream, rows))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    terms = torch.where((chosen >= E)[:, :, None], x.double()[:, None], y.double().view(n, top, dim))
    mixed = (weights.double()[:, :, None] * terms).sum(dim=1) + shared.double()
    want = x.double() + mixed / (mixed.square().mean(dim=1, keepdim=True) + 1e-5).sqrt() * gain.double()
    assert float((results[0][0].double() - want).norm() / want.norm()) < 2.0 ** -20
