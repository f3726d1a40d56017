"""32-bit linears of many rows by three bf16 parts: edges of tiles and of the parts of K, and numbers that three bf16 numbers cannot say."""

import pytest
import torch

from kestrel_amd.ops import core
from kestrel_amd.ops.linear import ACT_GATED, ACT_SILU

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _bound(a, w, extra=0.0):
    """Roundings of 2^-24 of the sum of magnitudes: 16 inside an instruction's sum, 8 within 128 of K, one per 128 of a quarter of K, the small products'
    (five per 16 of a quarter, each a 256th), four parts and four more at the end (what is left out is below one)."""
    k = a.shape[1]
    return (16 + 8 + k / 512 + 5 * k / 64 / 256 + 8) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + extra)


@pytest.mark.parametrize("m", [17, 31, 33, 65, 130, 300])
@pytest.mark.parametrize("n,k", [(1, 32), (33, 64), (70, 96), (130, 160), (64, 544), (2050, 2048), (515, 4128), (6200, 64), (40, 8192)])
def test_sums_at_edges(m, n, k):
    gen = torch.Generator(DEV).manual_seed(m * 131 + n + k)
    a = torch.randn(m, k + 4, generator=gen, device=DEV)[:, :k]
    w = torch.randn(n, k + 8, generator=gen, device=DEV)[:, 4:k + 4] * 0.05
    bias = torch.randn(n, generator=gen, device=DEV)
    out = torch.full((m, n + 1), 7.0, device=DEV)
    exact = a.double() @ w.double().T + bias.double()
    core.linear_generic(a, w, bias, out[:, :n])
    assert bool(((out[:, :n].double() - exact).abs() <= _bound(a, w, bias.double().abs())).all())
    assert bool((out[:, n] == 7.0).all())
    core.linear_generic(a, w, None, out[:, :n], accumulate=True)
    twice = exact * 2 - bias.double()
    assert bool(((out[:, :n].double() - twice).abs() <= 2 * _bound(a, w, bias.double().abs() + exact.abs())).all())


@pytest.mark.parametrize("m", [1, 16, 40])
def test_gated_pairs(m):
    gen = torch.Generator(DEV).manual_seed(m)
    a, w = torch.randn(m, 96, generator=gen, device=DEV), torch.randn(66, 96, generator=gen, device=DEV)
    out = torch.empty(m, 33, device=DEV)
    core.linear_generic(a, w, None, out, act=ACT_SILU | ACT_GATED)
    sums = a.double() @ w.double().T
    exact = torch.nn.functional.silu(sums[:, 0::2]) * sums[:, 1::2]
    # (silu's slope is at most 1.1; its own evaluation in fp32 a few roundings more)
    error = _bound(a, w)
    bound = 1.1 * error[:, 0::2] * sums[:, 1::2].abs() + (error[:, 1::2] + 8 * 2.0 ** -24 * sums[:, 1::2].abs()) * sums[:, 0::2].abs() + 1e-10
    assert bool(((out.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("scale", [1e-30, 1e-18, 1.0, 1e18, 3e37])
def test_scales_and_what_is_not_finite(scale):
    gen = torch.Generator(DEV).manual_seed(5)
    a, w = torch.rand(50, 256, generator=gen, device=DEV) - 0.5, (torch.rand(90, 256, generator=gen, device=DEV) - 0.5) * 0.02
    a *= scale
    w[3, 7] = 0.0
    a[4, 7], a[11, 200], a[12, 0], a[13, 0] = float("inf"), float("-inf"), float("nan"), 3.4e38          # (the last beyond bf16's largest)
    w[60, 9] = float("inf")
    out = torch.empty(50, 90, device=DEV)
    core.linear_generic(a, w, None, out)
    exact = a.double() @ w.double().T
    finite = exact.isfinite() & (exact.abs() < 3e38)
    assert bool((out.isnan() == exact.isnan()).all()) and bool((out.isinf() & (out > 0) == (exact == float("inf"))).all())
    assert bool(((out.double() - exact).abs() <= _bound(a, w) + 2.0 ** -126)[finite].all())


@pytest.mark.parametrize("m, n, k", [(17, 70, 32), (40, 70, 64), (40, 70, 160), (65, 2050, 544), (300, 520, 2048), (130, 260, 4128)])
@pytest.mark.parametrize("at", [0.0, 0.3, 1.0])
def test_weights_of_bf16_numbers(m, n, k, at):
    """Three products do where every weight of a part of K is a bf16 number: the same bits as six, which one weight of another kind asks for (``at``: where in K)."""
    gen = torch.Generator(DEV).manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=gen, device=DEV), torch.randn(n, k, generator=gen, device=DEV).bfloat16().float()
    out, other = torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
    core.linear_generic(a, w, None, out)
    assert bool(((out.double() - a.double() @ w.double().T).abs() <= _bound(a, w)).all())
    w[n // 2, int(at * (k - 1))] += 2.0 ** -20
    core.linear_generic(a, w, None, other)
    rest = torch.arange(n, device=DEV) != n // 2
    assert torch.equal(out[:, rest], other[:, rest])
    assert bool(((other.double() - a.double() @ w.double().T).abs() <= _bound(a, w)).all())
