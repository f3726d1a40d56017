"""The two last linears of a parallel block by tiles, K of both in parts, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _close_to_exact(got, terms, exact, extra=0.0):
    """A sum of products that are exact in 32 bits, added in any order: off by at most (terms) 2^-24 of the sum of magnitudes."""
    magnitudes, count = terms
    assert bool(((got.double().cpu() - exact).abs() <= count * 2.0 ** -24 * magnitudes + extra).all())


# rows and columns at the edges of tiles, parts inside either linear and across the border between them, one part, K of one step,
# the most tiles that are taken
@pytest.mark.parametrize("m, n, k1, k2", [(65, 128, 64, 64), (129, 516, 192, 1024), (128, 132, 1024, 192), (200, 2048, 2048, 1024),
                                          (300, 260, 64, 2048), (1280, 2048, 128, 576), (96, 20480, 64, 512), (70, 8192, 320, 512)])
@pytest.mark.parametrize("bias", [True, False])
def test_pair_by_tiles(m, n, k1, k2, bias):
    from kestrel_amd.ops import fast

    assert fast.pair_tile_parts(m, n, k1, k2) >= 1
    gen = torch.Generator().manual_seed(m + n + k1)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    a1, a2 = rnd(m, k1 + 8).bfloat16(), rnd(m, k2).bfloat16()
    w1, w2 = rnd(n, k1).bfloat16(), rnd(n, k2 + 16).bfloat16()
    b1, b2 = (rnd(n), rnd(n)) if bias else (None, None)
    x, gamma, beta = rnd(m, n), rnd(n), rnd(n)
    d = lambda t: t.to(DEV) if t is not None else None  # noqa: E731
    left = (d(a1)[:, :k1], d(w1), d(b1), d(a2), d(w2)[:, :k2], d(b2))
    exact = a1[:, :k1].double() @ w1.double().T + a2.double() @ w2[:, :k2].double().T
    terms = a1[:, :k1].double().abs() @ w1.double().abs().T + a2.double().abs() @ w2[:, :k2].double().abs().T
    if bias:
        exact, terms = exact + b1.double() + b2.double(), terms + b1.double().abs() + b2.double().abs()
    count = k1 + k2 + 3
    out = torch.full((m, n), float("nan"), device=DEV)
    assert fast.linear_pair_accumulate(*left, out, accumulate=False)
    _close_to_exact(out, (terms, count), exact)
    stream = d(x)
    assert fast.linear_pair_accumulate(*left, stream)
    _close_to_exact(stream, (terms + x.double().abs(), count), exact + x.double())
    normed = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    again = d(x)
    taken = fast.linear_pair_accumulate(*left, again, then_norm=(d(gamma), d(beta), 1e-5, normed))
    assert taken == (n <= 8192)
    if taken:
        assert torch.equal(again, stream)                # the same parts added in the same order
        want = torch.nn.functional.layer_norm(again.double().cpu(), (n,), gamma.double(), beta.double(), 1e-5)
        # statistics of 32 bits over the row (2^-16 of a number of the row covers them), then the rounding to bf16: half a step of 8 bits, 2^-8 of a number
        assert bool(((normed.double().cpu() - want).abs() <= (2.0 ** -8 + 2.0 ** -16) * want.abs() + 2.0 ** -14 * (1 + gamma.double().abs())).all())


# few rows: one row tile, weight tiles of 64 and of 128, parts in either linear and across the border
@pytest.mark.parametrize("m, n, k1, k2", [(17, 64, 64, 64), (33, 516, 192, 2048), (64, 2050, 2048, 320), (40, 8260, 320, 64), (64, 16400, 64, 512)])
def test_few_rows_of_a_pair_by_tiles(m, n, k1, k2):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + n + k1)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    a1, a2, w1, w2 = rnd(m, k1).bfloat16(), rnd(m, k2 + 8).bfloat16(), rnd(n, k1 + 8).bfloat16(), rnd(n, k2).bfloat16()
    x, bias = rnd(m, n), rnd(n)
    d = lambda t: t.to(DEV)  # noqa: E731
    stream = d(x)
    assert fast.linear_pair_accumulate(d(a1), d(w1)[:, :k1], d(bias), d(a2)[:, :k2], d(w2), None, stream)
    exact = a1.double() @ w1[:, :k1].double().T + a2[:, :k2].double() @ w2.double().T + bias.double() + x.double()
    terms = a1.double().abs() @ w1[:, :k1].double().abs().T + a2[:, :k2].double().abs() @ w2.double().abs().T + bias.double().abs() + x.double().abs()
    _close_to_exact(stream, (terms, k1 + k2 + 2), exact)


@pytest.mark.parametrize("m, n, k1, k2", [(64, 256, 64, 64), (65, 256, 72, 64), (65, 256, 64, 72), (65, 258, 64, 64), (1281, 2048, 128, 128)])
def test_what_is_not_taken_by_tiles(m, n, k1, k2):
    """Rows that the weight-streaming kernels take, K that is no multiple of a step, odd widths, more tiles than the rule allows."""
    from kestrel_amd.ops import fast

    assert fast.pair_tile_parts(m, n, k1, k2) == 0
    if m > fast.SKINNY_MAX_ROWS:
        bf = dict(dtype=torch.bfloat16, device=DEV)
        out = torch.zeros(m, n, device=DEV)
        assert not fast.linear_pair_accumulate(torch.zeros(m, k1, **bf), torch.zeros(n, k1, **bf), None, torch.zeros(m, k2, **bf),
                                               torch.zeros(n, k2, **bf), None, out)


def test_a_replayed_graph_repeats_the_eager_bits():
    from kestrel_amd.ops import fast

    torch.manual_seed(5)
    m, n, k1, k2 = 200, 512, 512, 2048
    bf = dict(dtype=torch.bfloat16, device=DEV)
    a1, a2, w1, w2 = torch.randn(m, k1, **bf), torch.randn(m, k2, **bf), torch.randn(n, k1, **bf), torch.randn(n, k2, **bf)
    eager, out = torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
    assert fast.linear_pair_accumulate(a1, w1, None, a2, w2, None, eager, accumulate=False)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fast.linear_pair_accumulate(a1, w1, None, a2, w2, None, out, accumulate=False)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert fast.linear_pair_accumulate(a1, w1, None, a2, w2, None, eager, accumulate=False)
