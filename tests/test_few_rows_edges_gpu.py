"""Linears of few rows where their launches differ: two targets of different kinds, K in no steps of 64, rows that are no numbers."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# K of 2,048: the persistent kernel; of 4,096 and 8,192: it too for few rows, else the split kernel up to 16 rows and one target after the
# other beyond
@pytest.mark.parametrize("persistent", [1, 0])
@pytest.mark.parametrize("k, hidden", [(2048, 704), (4096, 1792), (8192, 36), (1032, 8)])
@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 40, 64])
@pytest.mark.parametrize("columns", [33, 65])
def test_a_router_beside_a_gated_linear(columns, m, k, hidden, persistent):
    """Logits in fp32, an odd number of columns with a bias, beside the pairs of a gated bf16 linear. The bounds: a sum of K products is off
    by at most (K + 4) 2^-24 of their magnitudes; a gate's product of two such by that of either, and is rounded once (bf16 has eight bits: half
    a unit of the last is at most 2^-8)."""
    from kestrel_amd.ops import fast
    from kestrel_amd.ops.linear import ACT_GATED, activation_code

    gen = torch.Generator().manual_seed(columns + m + k)
    h, router = torch.randn(m, k, generator=gen).bfloat16(), (torch.randn(columns, k, generator=gen) * k ** -0.5).bfloat16()
    pairs, bias = (torch.randn(2 * hidden, k, generator=gen) * k ** -0.5).bfloat16(), torch.randn(columns, generator=gen)
    logits = torch.full((m, columns), float("nan"), device=DEV)
    out = torch.full((m, hidden), float("nan"), dtype=torch.bfloat16, device=DEV)
    fast.set_skinny_persistent(persistent)
    try:
        assert fast.linear_two_outputs(h.to(DEV), router.to(DEV), bias.to(DEV), logits, 0, pairs.to(DEV), None, out, activation_code("silu") | ACT_GATED)
    finally:
        fast.set_skinny_persistent(1)
    want = h.double() @ router.double().T + bias.double()
    slack = (k + 4) * 2.0 ** -24 * (h.double().abs() @ router.double().abs().T + bias.double().abs())
    assert bool(((logits.cpu().double() - want).abs() <= slack).all())
    z, s = ((a @ b.T).view(m, hidden, 2) for a, b in ((h.double(), pairs.double()), (h.double().abs(), (k + 4) * 2.0 ** -24 * pairs.double().abs())))
    gate = z[..., 0] * torch.sigmoid(z[..., 0])
    # (the gate's slope is at most 1.1, and its fast exponential and reciprocal are off by some 2^-21)
    slack = 1.1 * s[..., 0] * z[..., 1].abs() + gate.abs() * s[..., 1] + 1.001 * 2.0 ** -8 * (gate * z[..., 1]).abs() + 1e-6
    assert bool(((out.cpu().double() - gate * z[..., 1]).abs() <= slack).all())


@pytest.mark.parametrize("m", [17, 33, 48, 64])
@pytest.mark.parametrize("n, ks", [(1000, (8200,)), (8200, (4104,)), (2056, (2056, 8200)), (77, (2048, 8200)), (640, (72, 320))])
def test_wide_rows_of_a_length_in_no_steps_of_64(m, n, ks):
    """What is left to the kernel that holds activations in LDS, by the rule itself: every number of blocks of rows, many parts of K. fp32 sums."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + n)
    rows = [torch.randn(m, k, generator=gen).bfloat16() for k in ks]
    weights = [torch.randn(n, k, generator=gen).bfloat16() for k in ks]
    start = torch.randn(m, n, generator=gen)
    out = start.to(DEV)
    if len(ks) == 1:
        assert fast.linear_bf16(rows[0].to(DEV), weights[0].to(DEV), None, out, 0, True)
    else:
        assert fast.linear_pair_accumulate(rows[0].to(DEV), weights[0].to(DEV), None, rows[1].to(DEV), weights[1].to(DEV), None, out)
    want = start.double() + sum(a.double() @ w.double().T for a, w in zip(rows, weights))
    slack = (sum(ks) + 4) * 2.0 ** -24 * (start.double().abs() + sum(a.double().abs() @ w.double().abs().T for a, w in zip(rows, weights)))
    assert bool(((out.cpu().double() - want).abs() <= slack).all())


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_rows_that_are_no_numbers_stay_by_themselves(bad):
    """One number of one row, in every kernel of linears that tiles rows: all other rows are the same bits as without it."""
    from kestrel_amd.engine.batch import Workspace
    from kestrel_amd.ops import core, fast
    from kestrel_amd.ops.linear import ACT_GATED, activation_code

    gen = torch.Generator().manual_seed(5)
    act = activation_code("silu") | ACT_GATED

    def pair(a, m, n):
        out = torch.zeros(m, n, device=DEV)
        assert fast.linear_pair_accumulate(a[:, :192].contiguous(), w(n, 192), None, a[:, 192:].contiguous(), w(n, 256), None, out)
        return out

    def experts(a, m, n, few):
        y = torch.zeros(m * 2, 448, device=DEV)
        operands = (a, w(3, 128, 448), w(3, 448, 64), torch.arange(2 * m, dtype=torch.int32, device=DEV).view(m, 2) % 3)
        if few:
            assert fast.experts_few_bf16(*operands, torch.empty(m * 2, 64, dtype=torch.bfloat16, device=DEV), y, act)
        else:
            assert fast.experts_feed_forward_bf16(*operands, None, y, act, Workspace(torch.device(DEV)))
        return y.view(m, 2 * 448)

    def plain(a, m, n):
        out = torch.zeros(m, n, device=DEV)
        core.linear_generic(a.float(), w(n, 448).float(), None, out)
        return out

    def single(a, m, n):
        out = torch.zeros(m, n, device=DEV)
        assert fast.linear_bf16(a, w(n, 448), None, out, 0, True)
        return out

    def several(a, m, n):
        out = torch.zeros(m, n, dtype=torch.bfloat16, device=DEV)
        assert fast.linears_few_bf16([a, a], [w(n, 448), w(n, 448)], [torch.empty_like(out), out], (0, 0))
        return out

    weights = {}

    def w(*shape):
        if shape not in weights:
            weights[shape] = torch.randn(*shape, generator=gen).bfloat16().to(DEV)
        return weights[shape]

    for run, m, at in ((pair, 40, 17), (pair, 200, 130), (pair, 12, 11), (lambda *x: experts(*x, True), 40, 17), (lambda *x: experts(*x, False), 40, 17),
                       (lambda *x: experts(*x, False), 700, 300), (plain, 40, 17), (plain, 200, 60), (plain, 5, 2), (single, 33, 32), (several, 20, 3)):
        a = torch.randn(m, 448, generator=gen).bfloat16().to(DEV)
        clean = run(a, m, 320)
        assert bool(torch.isfinite(clean.float()).all())
        a[at, 7] = bad
        dirty = run(a, m, 320)
        others = torch.arange(m, device=DEV) != at
        assert torch.equal(clean[others], dirty[others]) and not bool(torch.isfinite(dirty[at].float()).any())
