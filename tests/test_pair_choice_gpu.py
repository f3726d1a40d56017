"""Two last linears of some hundred rows by either of their tiles, at the line between the small and the phased ones."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("m, n, k1, k2", [(400, 2048, 2048, 8192), (512, 2048, 2048, 8192), (576, 2048, 2048, 8192), (480, 2560, 2560, 10240),
                                          (512, 2560, 2560, 10240), (640, 2560, 2560, 2560), (900, 1024, 1024, 4096), (512, 4096, 4096, 8192)])
def test_small_and_phased_tiles(m, n, k1, k2):
    """Whichever of the two the estimate names, and the small tiles it would have without the phased ones: the sums are those of float64 to
    (K + 4) 2^-24 of their magnitudes."""
    from kestrel_amd.ops import fast

    handle, space = fast.lib(), fast._library_workspace(torch.device(DEV))
    codes = {fast.pair_tile_parts(m, n, k1, k2, phased) for phased in (False, True)}
    assert 0 not in codes and min(codes) < fast.PAIR_TILE_CODE
    gen = torch.Generator().manual_seed(m + n)
    a = [torch.randn(m, k, generator=gen).bfloat16().to(DEV) for k in (k1, k2)]
    w = [(torch.randn(n, k, generator=gen) * k ** -0.5).bfloat16().to(DEV) for k in (k1, k2)]
    start = torch.randn(m, n, generator=gen).to(DEV)
    want, size = start.double(), start.double().abs()
    for x, y in zip(a, w):
        want += x.double() @ y.double().T
        size += x.double().abs() @ y.double().abs().T
    ones, normed = torch.ones(n, device=DEV), torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    for code in sorted(codes):
        out = start.clone()
        fast._check(handle.ka_linear_pair_tiles_bf16(
            a[0].data_ptr(), k1, k1, a[1].data_ptr(), k2, k2, w[0].data_ptr(), k1, None, w[1].data_ptr(), k2, None, out.data_ptr(), n, n, 1, m, code,
            space.data_ptr(), space.numel() // 4, ones.data_ptr(), None, 1e-5, normed.data_ptr(), fast._OUT_CODE[normed.dtype], n, fast.stream_ptr()))
        assert bool(((out.double() - want).abs() <= (k1 + k2 + 4) * 2.0 ** -24 * size).all()), code
    out = start.clone()
    assert fast.linear_pair_accumulate(a[0], w[0], None, a[1], w[1], None, out)
    assert bool(((out.double() - want).abs() <= (k1 + k2 + 4) * 2.0 ** -24 * size).all())
