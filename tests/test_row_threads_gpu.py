"""Launches that finish whole rows of the stream, at every number of threads a row and pieces a thread, against float64."""

from __future__ import annotations

import pytest
import torch

from tests.plain import gozatar_plain as plain

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EPS = 1e-5


def _rel(got, want):
    return float((got.detach().double().cpu() - want).norm() / want.norm())


# (a thread per piece of few rows of 1,028 to 8,192 channels, several pieces a thread of many rows, the general form)
@pytest.mark.parametrize("n, dim", [(3, 1024), (3, 1028), (600, 2048), (7, 2048), (2, 4096), (530, 4096), (1, 5000), (3, 8192), (520, 8192), (4, 102)])
@pytest.mark.parametrize("top", [1, 6, 9])
def test_rows_are_finished(n, dim, top):
    """Sums of a handful of fp32 terms and of squares over a row: 2^-20 in the 2-norm; what is rounded to bf16 is off by at most 2^-8 of a number."""
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(n + dim + top)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    E = 5
    chosen = torch.randint(0, E + 2, (n, top), generator=gen).to(torch.int32)          # (from E on: the input itself)
    weights, y, h, shared, sg = torch.rand(n, top, generator=gen), rnd(n * top, dim), rnd(n, dim).bfloat16(), rnd(n, dim), rnd(n)
    gain, gain2, x = 1 + 0.2 * rnd(dim), 1 + 0.2 * rnd(dim), rnd(n, dim)
    own = chosen.view(-1) >= E
    y[own] = float("nan")                                                              # (rows that nobody has written)
    terms = torch.where(own[:, None], h.double().repeat_interleave(top, 0), y.double()).view(n, top, dim)
    mixed = (weights.double()[:, :, None] * terms).sum(dim=1) + torch.sigmoid(sg.double())[:, None] * shared.double()
    stream = x.double() + plain.rms(mixed, EPS) * gain.double()
    operands = (y.to(DEV), h.to(DEV), chosen.to(DEV), weights.to(DEV), E, shared.to(DEV), sg.to(DEV))
    for then in (None, (gain2.to(DEV), EPS)):
        for rows in (None, torch.full((n, dim), float("nan"), dtype=torch.bfloat16, device=DEV)):
            if then is not None and rows is None:
                continue
            got = x.to(DEV)
            core.experts_combine_normed(*operands, got, (gain.to(DEV), EPS), then, rows)
            again, left = x.to(DEV), None if rows is None else torch.full_like(rows, float("nan"))
            core.add_normed(again, mixed.float().to(DEV), (gain.to(DEV), EPS), then, left)
            assert _rel(got, stream) < 2.0 ** -20 and _rel(again, stream) < 2.0 ** -20
            if rows is not None:
                want = stream if then is None else plain.rms(stream, EPS) * gain2.double()
                assert bool(((rows.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all())
                assert bool(((left.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all())
    S = 1 + (n + top) % 4
    streams, mix, out, into = rnd(n, S, dim), rnd(S, S), rnd(S), torch.rand(S, generator=gen) + 0.2
    want = plain.write_streams(streams.transpose(0, 1).double(), mix.double(), out.double(), mixed)
    read = plain.layer_norm(plain.read_streams(want, into.double()), gain.double(), EPS)
    reading = (into.to(DEV), ("layernorm", gain.to(DEV), None, EPS))
    got, rows = streams.to(DEV), torch.full((n, dim), float("nan"), device=DEV)
    core.streams_experts(got, operands[0], h.float().to(DEV), *operands[2:], mix.to(DEV), out.to(DEV), reading, rows)
    again, left = streams.to(DEV), torch.full((n, dim), float("nan"), device=DEV)
    core.streams_step(again, mixed.float().to(DEV), mix.to(DEV), out.to(DEV), reading, left)
    for x_, r_ in ((got, rows), (again, left)):
        assert _rel(x_.transpose(0, 1), want) < 2.0 ** -19 and _rel(r_, read) < 2.0 ** -18
