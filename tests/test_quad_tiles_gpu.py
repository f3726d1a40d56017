"""Linears of prompts by four waves a tile: one linear and two of the same rows, against float64; where they go there."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TILES = (3, 5, 6, 7, 8, 9, 10, 11, 12)


def _close(got, want, magnitudes, count, rounded):
    """As in ``test_phased_tiles_gpu.py``: sums in 32 bits in any order, the rounding to bf16, an activation of slope at most 1.13."""
    bound = 1.13 * (count + 8) * 2.0 ** -24 * magnitudes + (2.0 ** -8 * want.abs() if rounded else 0.0)
    assert bool(((got.double() - want).abs() <= bound + 2.0 ** -60).all())


# every tile: one K-step, as many as there are stages and one more or less, many; rows and columns at the edges of tiles and of the waves' quarters
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m, n, k", [(1, 8, 64), (129, 264, 128), (97, 200, 192), (300, 72, 256), (193, 520, 320), (512, 640, 1344)])
def test_one_linear(tile, m, n, k):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + n + k)
    a, w, b = (torch.randn(*s, generator=gen) for s in ((m, k + 8), (n, k + 16), (n,)))
    a, w, b, start = a.bfloat16().to(DEV), w.bfloat16().to(DEV), b.to(DEV), torch.randn(m, n + 8, generator=gen).to(DEV)
    x, y = a[:, :k].double(), w[:, :k].double()
    want, size = x @ y.T, x.abs() @ y.abs().T
    for dtype, bias, act, acc in ((torch.bfloat16, b, 0, 0), (torch.bfloat16, None, 1, 0), (torch.float32, b, 3, 0), (torch.float32, None, 0, 1)):
        out = start.to(dtype, copy=True)
        fast._check(fast.lib().ka_linear_quad_bf16(a.data_ptr(), k + 8, w.data_ptr(), k + 16, fast._ptr(bias), out.data_ptr(), fast._OUT_CODE[dtype], n + 8, m, n, k, act, acc,
                                                   tile, torch.cuda.current_stream().cuda_stream))
        z, s = (want, size) if bias is None else (want + b.double(), size + b.double().abs())
        z = torch.nn.functional.gelu(z, approximate="tanh") if act == 1 else torch.nn.functional.silu(z) if act == 3 else z
        if acc:
            z, s = z + start[:, :n].double(), s + start[:, :n].double().abs()
        _close(out[:, :n], z, s, k + 2, dtype == torch.bfloat16)
        assert torch.equal(out[:, n:], start[:, n:].to(dtype))


@pytest.mark.parametrize("tile", TILES)
def test_two_linears(tile):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(tile)
    m, n1, n2, k = 261, 136, 424, 448
    a, w1, w2, b = (torch.randn(*s, generator=gen) for s in ((m, k), (n1, k), (n2, k), (n2,)))
    a, w1, w2, b = a.bfloat16().to(DEV), w1.bfloat16().to(DEV), w2.bfloat16().to(DEV), b.to(DEV)
    outs = [torch.full((m, n + 8), 7.0, dtype=torch.bfloat16, device=DEV) for n in (n1, n2)]
    fast._check(fast.lib().ka_linear_joint_bf16(a.data_ptr(), k, m, k, w1.data_ptr(), k, None, outs[0].data_ptr(), n1 + 8, n1, 1, w2.data_ptr(), k, b.data_ptr(),
                                                outs[1].data_ptr(), n2 + 8, n2, 0, tile, torch.cuda.current_stream().cuda_stream))
    x, y, z = a.double(), w1.double(), w2.double()
    _close(outs[0][:, :n1], torch.nn.functional.gelu(x @ y.T, approximate="tanh"), x.abs() @ y.abs().T, k, True)
    _close(outs[1][:, :n2], x @ z.T + b.double(), x.abs() @ z.abs().T + b.double().abs(), k + 1, True)
    assert all(bool((o[:, n:] == 7.0).all()) for o, n in zip(outs, (n1, n2)))


def test_where_a_linear_goes():
    """One round of tiles that are enough for the length of K; what the tiles do not cover stays where it was, with the same result."""
    from kestrel_amd.ops import fast

    rule = lambda m, n, k: fast.lib().ka_linear_quad_tile(m, n, k)  # noqa: E731
    assert [rule(*s) for s in ((2048, 2048, 2048), (512, 5632, 2048), (256, 2048, 2048), (80, 3072, 1024), (80, 512, 1024), (768, 4096, 4096), (768, 2048, 4096), (1024, 2048, 8192),
                               (2048, 6144, 2048), (300, 2048, 72), (300, 2052, 128))] == [8, 7, 0, 6, 0, 0, 6, 0, 0, 0, 0]
    gen = torch.Generator().manual_seed(1)
    a, w = torch.randn(300, 512, generator=gen).bfloat16().to(DEV), torch.randn(2048, 512, generator=gen).bfloat16().to(DEV)
    bias = torch.randn(2049, generator=gen).to(DEV)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    for b, columns, n in ((None, 2048, 2048), (bias[1:], 2048, 2048), (None, 2052, 2048), (None, 2048, 2044)):   # (a bias off its alignment, rows and outputs in no eights)
        out = torch.full((300, columns), 7.0, device=DEV)
        assert fast.linear_bf16(a, w[:n], b[:n] if b is not None else None, out[:, :n], 0, False)
        _close(out[:, :n], want[:, :n] + (0 if b is None else b.double()), size[:, :n] + (0 if b is None else b.double().abs()), 513, False)
        assert bool((out[:, n:] == 7.0).all())
