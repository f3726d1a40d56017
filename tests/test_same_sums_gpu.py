"""Sums whose order is the same whatever tile, number of threads or kernel a step's size calls for: equal bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("n, dim, ff", [(1, 80, 16), (150, 208, 80), (257, 144, 336)])
def test_listed_experts_do_not_depend_on_the_tile(n, dim, ff, gated):
    """The kernel for sizes in no steps of 64 and the tiles for those that are, the same operands with zeros behind their last channel."""
    from kestrel_amd.engine.batch import Workspace
    from kestrel_amd.ops import fast
    from kestrel_amd.ops.linear import ACT_GATED, activation_code

    gen = torch.Generator().manual_seed(n + dim + ff)
    n_experts, top = 5, 3
    act = activation_code("silu") | ACT_GATED if gated else activation_code("relu_squared")
    h = torch.randn(n, dim, generator=gen).bfloat16()
    first = (torch.randn(n_experts, ff * (2 if gated else 1), dim, generator=gen) * dim ** -0.5).bfloat16()
    down = (torch.randn(n_experts, dim, ff, generator=gen) * ff ** -0.5).bfloat16()
    chosen = torch.stack([torch.randperm(n_experts, generator=gen)[:top] for _ in range(n)]).to(torch.int32).to(DEV)
    dim64, ff64 = -(-dim // 64) * 64, -(-ff // 64) * 64
    assert dim64 > dim and ff64 > ff
    pad = lambda t, *sizes: torch.nn.functional.pad(t, [x for have, want in zip(reversed(t.shape), reversed(sizes)) for x in (0, want - have)])  # noqa: E731
    results = []
    for operands, width, tiles in (((h, first, down), dim, (128,)),
                                   ((pad(h, n, dim64), pad(first, n_experts, first.shape[1] // ff * ff64, dim64), pad(down, n_experts, dim64, ff64)), dim64,
                                    (64, 128, 256))):
        for tile in tiles:
            y = torch.full((n * top, width), float("nan"), device=DEV)
            assert fast.experts_feed_forward_bf16(*(t.to(DEV) for t in operands), chosen, None, y, act, Workspace(torch.device(DEV)), tile=tile)
            results.append(y[:, :dim].cpu())
    assert all(torch.equal(results[0], other) for other in results[1:])


@pytest.mark.parametrize("dim", [1028, 2048, 2560, 4096, 5000, 8192])
def test_rows_of_the_stream_do_not_depend_on_their_number(dim):
    """Many rows get 256 threads each, few get one a piece: the numbers of a row are the same bits."""
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(dim)
    n, few, top, E, S = 1100, 5, 4, 6, 4                       # (1,100: more than two rows a CU)
    rnd = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)  # noqa: E731
    streams, x, y, h, shared = rnd(n, S, dim), rnd(n, dim), rnd(n * top, dim), rnd(n, dim).bfloat16(), rnd(n, dim)
    chosen = torch.randint(0, E + 1, (n, top), generator=gen).to(torch.int32).to(DEV)
    weights, mix, out, into, gain, gain2 = rnd(n, top).abs(), rnd(S, S), rnd(S), rnd(S), rnd(dim), rnd(dim)

    def results(m):
        done = []
        for kind in ("layernorm", "rms"):
            got, rows = streams[:m].clone(), torch.full((m, dim), float("nan"), device=DEV)
            core.streams_step(got, x[:m].contiguous(), mix, out, (into, (kind, gain, None, 1e-5)), rows)
            again, left = streams[:m].clone(), torch.full((m, dim), float("nan"), device=DEV)
            core.streams_experts(again, y[:m * top], h[:m].float(), chosen[:m], weights[:m], E, shared[:m], None, mix, out,
                                 (into, (kind, gain, None, 1e-5)), left)
            done += [got, rows, again, left]
        got, rows = x[:m].clone(), torch.full((m, dim), float("nan"), dtype=torch.bfloat16, device=DEV)
        core.experts_combine_normed(y[:m * top], h[:m], chosen[:m], weights[:m], E, shared[:m], None, got, (gain, 1e-5), (gain2, 1e-5), rows)
        again, left = x[:m].clone(), torch.full((m, dim), float("nan"), device=DEV)
        core.add_normed(again, shared[:m].contiguous(), (gain, 1e-5), (gain2, 1e-5), left)
        return [t[:few].cpu() for t in done + [got, rows, again, left]]

    for i, (a, b) in enumerate(zip(results(n), results(few))):
        assert torch.equal(a, b), f"result {i}"
