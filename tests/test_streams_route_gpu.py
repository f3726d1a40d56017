"""The step between sublayers with a router's linear and its choice in the same launch: the step's own bits, the logits, and the choice by them."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# (a thread a piece, 512 and 1,024 of them: the shortest and longest rows of either, and ends inside a wave's load; outputs of one wave each and more rounds than
# are asked for ahead; a row of the linear that is not chosen among)
@pytest.mark.parametrize("n, S, dim, outputs, more", [(1, 4, 2048, 30, 0), (7, 4, 1032, 1, 0), (64, 3, 2056, 64, 1), (40, 4, 4096, 62, 0), (3, 2, 4088, 33, 64), (2, 1, 2048, 8, 0)])
def test_step_and_choice(n, S, dim, outputs, more):
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(n + dim + outputs)
    rnd = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)  # noqa: E731
    x, y, mix, out, into, gain, shift = rnd(n, S, dim), rnd(n, dim), rnd(S, S), rnd(S), rnd(S), rnd(dim), rnd(dim)
    router = torch.full((outputs + more, dim + 8), 7.0, dtype=torch.bfloat16, device=DEV)[:, :dim]       # (columns of wider rows)
    router.copy_(rnd(outputs + more, dim) * dim ** -0.5)
    groups, top = (2, 2) if outputs % 2 == 0 else (0, 1)
    for bias, correction, form, options in ((None, rnd(outputs) * 0.1, ("layernorm", gain, shift, 1e-5), dict(scores="sigmoid", group_best=2, always=99)),
                                            (rnd(outputs + more), None, ("rms", gain, None, 1e-5), dict(weigh_chosen=True))):
        kept = (0, 0) if options.get("weigh_chosen") else (groups, 1 if groups else 0)
        columns = top + ("always" in options)
        want_x, want_h = x.clone(), torch.empty(n, dim, dtype=torch.bfloat16, device=DEV)
        core.streams_step(want_x, y, mix, out, (into, form), want_h)
        got_x, h = x.clone(), torch.empty(n, dim, dtype=torch.bfloat16, device=DEV)
        logits = torch.full((n, outputs + more + 3), 7.0, device=DEV)
        chosen, weights = torch.full((n, columns), -1, dtype=torch.int32, device=DEV), torch.full((n, columns), 7.0, device=DEV)
        choice = (outputs, correction, top, *kept, 2.5)
        assert core.streams_step_route(got_x, y, mix, out, (into, form), h, router, bias, logits, *choice, chosen, weights, **options)
        assert torch.equal(got_x, want_x) and torch.equal(h, want_h)
        assert bool((logits[:, outputs + more:] == 7.0).all())
        want = h.double() @ router.double().T + (0 if bias is None else bias.double())
        # (sums of at most 4,096 products, none more than 2^-24 of the sum of their sizes off per addition; the chains are of 8 and 64 lanes are added in pairs)
        room = (h.double().abs() @ router.double().abs().T + 1) * 24 * 2.0 ** -24
        assert bool(((logits[:, :outputs + more].double() - want).abs() <= room).all())
        again, again_weights = torch.empty_like(chosen), torch.empty_like(weights)
        core.route(logits[:, :outputs + more], *choice, again, again_weights, **options)
        assert torch.equal(chosen, again) and torch.equal(weights, again_weights)
        one_x, one_h, one = x[n - 1:].clone(), torch.empty(1, dim, dtype=torch.bfloat16, device=DEV), torch.empty(1, outputs + more, device=DEV)
        assert core.streams_step_route(one_x, y[n - 1:].contiguous(), mix, out, (into, form), one_h, router, bias, one, *choice, again[:1].clone(),
                                       again_weights[:1].clone(), **options)
        assert torch.equal(one[0], logits[n - 1, :outputs + more])


def test_what_stays_with_two_launches():
    """Short and long rows, five streams, more outputs than a wave, a 32-bit router: nothing is run."""
    from kestrel_amd.ops import core

    for S, dim, outputs, dtype in ((4, 1024, 8, torch.bfloat16), (4, 4104, 8, torch.bfloat16), (5, 2048, 8, torch.bfloat16), (4, 2048, 65, torch.bfloat16),
                                   (4, 2048, 8, torch.float32), (4, 2052, 8, torch.bfloat16)):
        x, y, h = torch.ones(2, S, dim, device=DEV), torch.ones(2, dim, device=DEV), torch.full((2, dim), 7.0, dtype=torch.bfloat16, device=DEV)
        form = (None, ("rms", torch.ones(dim, device=DEV), None, 1e-5))
        router, logits = torch.ones(outputs, (dim + 7) // 8 * 8, dtype=dtype, device=DEV)[:, :dim], torch.empty(2, outputs, device=DEV)
        chosen, weights = torch.empty(2, 1, dtype=torch.int32, device=DEV), torch.empty(2, 1, device=DEV)
        assert not core.streams_step_route(x, y, torch.ones(S, S, device=DEV), torch.ones(S, device=DEV), form, h, router, None, logits, outputs, None, 1, 0, 0, 1.0,
                                           chosen, weights)
        assert bool((x == 1.0).all()) and bool((h == 7.0).all())


# (one row, either side of 16 and of the most rows that stream weights; rows of 2,048 and the next longer ones, of 2,560 and the next; a shared expert among the others, of its own, none)
@pytest.mark.parametrize("n", [1, 16, 17, 64, 65])
@pytest.mark.parametrize("dim, shared", [(2048, "joined"), (2048, "own"), (2048, None), (2112, "joined"), (2560, "joined"), (2624, "joined"), (4096, "own")])
def test_where_the_choice_goes(n, dim, shared):
    """A routed mixture behind streams: the choice in the step's launch or in its own, by rows, width and shared expert; the same experts either way, and the same streams but for roundings."""
    from types import SimpleNamespace

    from kestrel_amd.engine.batch import Workspace
    from kestrel_amd.ops import core
    from kestrel_amd.parts.experts import RoutedExperts
    from kestrel_amd.parts.specs import RoutedExpertsSpec

    gen = torch.Generator().manual_seed(n + dim)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    spec = RoutedExpertsSpec("routed_experts", dim, 6, 64, 2, scores="sigmoid", group_best=2, shared_hidden={"joined": 64, "own": 128, None: None}[shared], shared_gate=False)
    part = RoutedExperts(spec)
    weights = {name: (rnd(*p.shape) * (p.shape[-1] ** -0.5 if len(p.shape) > 1 else 0.1)).bfloat16() for name, p in part.params().items()}
    part.bind(weights, torch.bfloat16, torch.device(DEV))
    streams = SimpleNamespace(matrix=rnd(3, 3).to(DEV), out=rnd(3).to(DEV))
    reading = (rnd(3).to(DEV), ("rms", rnd(dim).to(DEV), None, 1e-5))
    x, y = rnd(n, 3, dim).to(DEV), rnd(n, dim).to(DEV)
    results = []
    for together in (True, False):
        batch, rows, h = SimpleNamespace(workspace=Workspace(torch.device(DEV))), x.clone(), torch.full((n, dim), 7.0, dtype=torch.bfloat16, device=DEV)
        took = together and part.choose_streams(rows, y, streams, reading, h, batch)
        assert took == (together and n <= 64 and (dim == 2048 and shared != "own" or dim > 2560 and n > 16))
        if not took:
            assert torch.equal(rows, x) and bool((h == 7.0).all())
            core.streams_step(rows, y, streams.matrix, streams.out, reading, h)
        part.mix_streams(h, batch, rows, streams, None, None, chosen=took)
        results.append((h, batch.workspace.get("experts.chosen", (n, 2 + part.joined), torch.int32).clone(), rows))
    (h, chosen, rows), (want_h, want_chosen, want_rows) = results
    assert torch.equal(h, want_h) and torch.equal(chosen.sort(dim=1).values, want_chosen.sort(dim=1).values)
    # (the weights of a choice differ by the order of the router's sums, some 24 roundings of 2^-24; a sigmoid's slope is a quarter)
    assert bool(((rows - want_rows).abs() <= 1e-4 * want_rows.abs().amax(dim=(1, 2), keepdim=True)).all())
