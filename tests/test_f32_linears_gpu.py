"""The 32-bit linears at the edges of their tiles, parts and columns, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _operands(m, n, k, seed, lda=None):
    gen = torch.Generator().manual_seed(seed)
    a = torch.randn(m, lda or k, generator=gen).to(DEV)[:, :k]
    return a, torch.randn(n, k, generator=gen).to(DEV), torch.randn(n, generator=gen).to(DEV)


# one row to sixteen (a wave per column), then tiles of 32 x 32 to 64 x 128; columns that end inside a wave's, a tile's and a
# vector's; K of one step of 32, of fewer steps than parts, of parts that differ in length, of steps that are cut short
@pytest.mark.parametrize("m, n, k", [(1, 5, 36), (3, 4097, 1028), (4, 9000, 2048), (7, 130, 4100), (16, 8200, 1024), (17, 1, 32), (17, 33, 64),
                                     (40, 2048, 96), (33, 131, 160), (157, 6146, 288), (300, 8192, 64), (130, 1000, 2080), (1500, 2050, 128), (2100, 4096, 32)])
def test_f32_linears(m, n, k):
    """Bound: a sum of K products is off by at most (K + 4) 2^-24 of the sum of their magnitudes (and less by far)."""
    from kestrel_amd.ops import core

    a, w, bias = _operands(m, n, k, m + n + k, lda=k + 4)
    want = a.double() @ w.double().T
    slack = (k + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs())
    out = torch.full((m, n + 3), 5.0, device=DEV)
    core.linear_generic(a, w, bias, out[:, :n])
    assert bool(((out[:, :n].double() - want - bias.double()).abs() <= slack).all()) and bool((out[:, n:] == 5.0).all())
    out = torch.ones(m, n, device=DEV)
    core.linear_generic(a, w, None, out, accumulate=True)
    assert bool(((out.double() - want - 1.0).abs() <= slack + 2.0 ** -23 * want.abs()).all())
    out = torch.zeros(m, n, device=DEV)
    core.linear_generic(a, w, bias, out, act=2)
    assert bool(((out.double() - (want + bias.double()).clamp(min=0.0)).abs() <= slack).all())
    if n % 2 == 0:
        out = torch.zeros(m, n // 2, device=DEV)
        core.linear_generic(a, w, bias, out, act=2 | 0x100)
        full, s = want + bias.double(), slack
        gate = full[:, 0::2].clamp(min=0.0)
        assert bool(((out.double() - gate * full[:, 1::2]).abs() <= 1.01 * (s[:, 0::2] * full[:, 1::2].abs() + gate * s[:, 1::2]) + 1e-6).all())


@pytest.mark.parametrize("k", [32, 160, 2048])
def test_a_row_has_the_same_bits_in_every_tile(k):
    """The order of a row's sums is fixed by K: alone with sixteen others, in a hundred or in two thousand rows."""
    from kestrel_amd.ops import core

    a, w, bias = _operands(2050, 4100, k, k)
    whole = torch.empty(2050, 4100, device=DEV)
    core.linear_generic(a, w, bias, whole)
    for rows in (17, 40, 157, 303, 1100):
        part = torch.empty(rows, 4100, device=DEV)
        core.linear_generic(a[:rows], w, bias, part)
        assert torch.equal(part, whole[:rows]), rows
        narrow = torch.empty(rows, 260, device=DEV)
        core.linear_generic(a[:rows], w[:260], bias[:260], narrow)
        assert torch.equal(narrow, whole[:rows, :260]), rows
