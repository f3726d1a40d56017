"""32-bit linears of many rows on the matrix pipes, in 32 bits and by three bf16 parts: edges of tiles and of the parts of K, and numbers that three bf16 numbers cannot say."""

import pytest
import torch

from kestrel_amd.ops import core
from kestrel_amd.ops.linear import ACT_GATED, ACT_SILU

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _bound(a, w, extra=0.0):
    """Roundings of 2^-24 of the sum of magnitudes. Three parts: 16 inside an instruction's sum, 8 within 128 of K, one per 128 of a quarter of K, the small products' (two per
    16 of a quarter, each a 256th), four parts and four more at the end. In 32 bits: 16 within 16 of K, one per 16 of a quarter of K, the same at the end."""
    k = a.shape[1]
    return max(16 + 8 + k / 512 + 2 * k / 64 / 256 + 8, 16 + k / 64 + 8) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + extra)


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
@pytest.mark.parametrize("kind", ["bf16", "32 bits"])
def test_scales_and_what_is_not_finite(scale, kind):
    gen = torch.Generator(DEV).manual_seed(5)
    a, w = torch.rand(50, 256, generator=gen, device=DEV) - 0.5, (torch.rand(90, 256, generator=gen, device=DEV) - 0.5) * 0.02
    w = w.bfloat16().float() if kind == "bf16" else w
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
    """Weights that are bf16 numbers: the activations' three parts; one weight of another kind (``at``: where in K) changes its own output alone."""
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


@pytest.mark.parametrize("k", [32, 160, 2048])
@pytest.mark.parametrize("every", [0, 3, 64])
def test_a_row_has_the_same_bits_beside_any_others(k, every):
    """bf16 weights, and rows of them of 32 bits between: alone with sixteen others, in a hundred, in a thousand rows, and beside other outputs."""
    gen = torch.Generator(DEV).manual_seed(k + every)
    a, w = torch.randn(1100, k, generator=gen, device=DEV), torch.randn(4100, k, generator=gen, device=DEV).bfloat16().float()
    if every:
        w[::every] = torch.randn_like(w[::every])
    a[7] *= 1e-35
    whole = torch.empty(1100, 4100, device=DEV)
    core.linear_generic(a, w, None, whole)
    assert bool(((whole.double() - a.double() @ w.double().T).abs() <= _bound(a, w)).all())
    for rows in (17, 40, 157, 303):
        for first, last in ((0, 4100), (31, 290)):
            part = torch.empty(rows, last - first, device=DEV)
            core.linear_generic(a[:rows], w[first:last], None, part)
            assert torch.equal(part, whole[:rows, first:last])


@pytest.mark.parametrize("m", [40, 300])
@pytest.mark.parametrize("kind", ["bf16", "32 bits"])
@pytest.mark.parametrize("x_scale, w_scale", [(1e-33, 1.0), (1e-35, 1.0), (7.5e-37, 1.0), (1.0, 1e-33), (1.0, 1e-36), (1e-35, 1e33), (1e33, 1e-35)])
def test_numbers_whose_third_part_bf16_does_not_hold(m, kind, x_scale, w_scale):
    """Numbers below 2^-109 have bits below bf16's smallest: every third row of either operand is of such numbers, and their sums are as good as any other (a product's own
    last place is 2^-149 at the least). The rows beside them have the bits they have without."""
    gen = torch.Generator(DEV).manual_seed(m)
    a, w = torch.randn(m, 544, generator=gen, device=DEV), torch.randn(130, 544, generator=gen, device=DEV) * 0.05
    rows, columns = torch.arange(m, device=DEV) % 3 == 1, torch.arange(130, device=DEV) % 3 == 2
    as_kind = lambda t: t.bfloat16().float() if kind == "bf16" else t  # noqa: E731
    w = as_kind(w)
    plain = torch.empty(m, 130, device=DEV)
    core.linear_generic(a, w, None, plain)
    a[rows] *= x_scale
    w[columns] = as_kind(w[columns] * w_scale)
    out = torch.empty(m, 130, device=DEV)
    core.linear_generic(a, w, None, out)
    assert bool(((out.double() - a.double() @ w.double().T).abs() <= _bound(a, w) + 544 * 2.0 ** -149).all())
    same = ~((rows & (x_scale != 1.0))[:, None] | (columns & (w_scale != 1.0))[None, :])
    assert torch.equal(out[same], plain[same])


@pytest.mark.parametrize("m", [33, 300])
@pytest.mark.parametrize("kind", ["bf16", "32 bits"])
def test_a_sum_of_one_product(m, kind):
    """One product alone: its own rounding to 24 bits and, for the small products of a bf16 weight, which weigh 2^-8, theirs."""
    gen = torch.Generator(DEV).manual_seed(m)
    a, w = torch.zeros(m, 160, device=DEV), torch.rand(515, 160, generator=gen, device=DEV) + 1
    w = w.bfloat16().float() if kind == "bf16" else w
    a[torch.arange(m, device=DEV), torch.arange(m, device=DEV) % 160] = torch.rand(m, generator=gen, device=DEV) + 1
    out = torch.empty(m, 515, device=DEV)
    core.linear_generic(a, w, None, out)
    exact = a.double() @ w.double().T
    assert float(((out.double() - exact) / exact).abs().max()) <= 2.0 ** -24 * (1 + 2 * 2.0 ** -8)


def test_not_a_number_in_every_row_costs_a_pass_of_products():
    """Such sums are multiplied once more by products of 32 bits, not one output after another (some 1.8 times the usual time)."""
    gen = torch.Generator(DEV).manual_seed(1)
    a, w = torch.randn(300, 2048, generator=gen, device=DEV), torch.randn(2048, 2048, generator=gen, device=DEV).bfloat16().float()
    out = torch.empty(300, 2048, device=DEV)

    def best():
        times = []
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            core.linear_generic(a, w, None, out)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    usual = best()
    a[:, 5] = float("nan")
    assert best() < 8 * usual and bool(out.isnan().all())
