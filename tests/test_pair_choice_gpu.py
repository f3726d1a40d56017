"""Which tiles two last linears of some hundred rows get, at the line between the small and the phased ones."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("m, n, k1, k2, tile", [(400, 2048, 2048, 8192, 3), (512, 2048, 2048, 8192, 3), (576, 2048, 2048, 8192, 0), (480, 2560, 2560, 10240, 3),
                                                (512, 2560, 2560, 10240, 3), (640, 2560, 2560, 2560, 3), (900, 1024, 1024, 4096, 0), (512, 4096, 4096, 8192, 1)])
def test_small_or_phased_tiles(m, n, k1, k2, tile):
    """The line lies where both take as long; on either side of it the sums are those of float64 to (K + 4) 2^-24 of their magnitudes."""
    from kestrel_amd.ops import fast

    assert fast.pair_tile_parts(m, n, k1, k2) // fast.PAIR_TILE_CODE == tile
    gen = torch.Generator().manual_seed(m + n)
    a = [torch.randn(m, k, generator=gen).bfloat16().to(DEV) for k in (k1, k2)]
    w = [(torch.randn(n, k, generator=gen) * k ** -0.5).bfloat16().to(DEV) for k in (k1, k2)]
    start = torch.randn(m, n, generator=gen).to(DEV)
    out = start.clone()
    assert fast.linear_pair_accumulate(a[0], w[0], None, a[1], w[1], None, out)
    want, size = start.double(), start.double().abs()
    for x, y in zip(a, w):
        want += x.double() @ y.double().T
        size += x.double().abs() @ y.double().abs().T
    assert bool(((out.double() - want).abs() <= (k1 + k2 + 4) * 2.0 ** -24 * size).all())
