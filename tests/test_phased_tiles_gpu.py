"""Two last linears of prompts on the phased tiles, K of both in parts, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _rnd(seed):
    gen = torch.Generator().manual_seed(seed)
    return lambda *shape: torch.randn(*shape, generator=gen)


def _close(got, want, magnitudes, count):
    """A sum of ``count`` products that are exact in 32 bits, in any order, is off by at most count 2^-24 of the sum of magnitudes."""
    bound = count * 2.0 ** -24 * magnitudes
    assert bool(((got.double().cpu() - want).abs() <= bound).all())


# every tile of it: one part and several, the border between the linears at a part's start, inside one, behind an odd number of K-steps
@pytest.mark.parametrize("tile", [0, 1, 3])
@pytest.mark.parametrize("m, n, k1, k2, parts", [(65, 132, 64, 64, 1), (257, 260, 192, 1024, 3), (300, 516, 512, 512, 2), (513, 128, 640, 320, 7), (256, 256, 1088, 64, 2)])
def test_two_last_linears_in_parts(tile, m, n, k1, k2, parts):
    from kestrel_amd.ops import fast

    rnd = _rnd(m + n + parts)
    a1, a2, w1, w2, b1, b2, x = rnd(m, k1 + 8).bfloat16(), rnd(m, k2).bfloat16(), rnd(n, k1).bfloat16(), rnd(n, k2 + 8).bfloat16(), rnd(n), rnd(n), rnd(m, n)
    d = [t.to(DEV) for t in (a1, a2, w1, w2, b1, b2)]
    out = x.to(DEV)
    space = fast._library_workspace(out.device)
    fast._check(fast.lib().ka_linear_pair_tiles_bf16(
        d[0].data_ptr(), k1 + 8, k1, d[1].data_ptr(), k2, k2, d[2].data_ptr(), k1, d[4].data_ptr(), d[3].data_ptr(), k2 + 8, d[5].data_ptr(),
        out.data_ptr(), n, n, 1, m, parts + fast.PAIR_TILE_CODE * tile, space.data_ptr(), space.numel() // 4, None, None, 0.0, None, 0, 0,
        torch.cuda.current_stream().cuda_stream))
    p, q, r, s = a1[:, :k1].double(), w1.double(), a2.double(), w2[:, :k2].double()
    rest = b1.double() + b2.double() + x.double()
    _close(out, p @ q.T + r @ s.T + rest, p.abs() @ q.abs().T + r.abs() @ s.abs().T + b1.double().abs() + b2.double().abs() + x.double().abs(), k1 + k2 + 3)


@pytest.mark.parametrize("m, n, k1, k2, large", [(1280, 2048, 2048, 8192, False), (1281, 2048, 2048, 8192, True), (2048, 2048, 2048, 8192, True),
                                                 (2048, 2048, 512, 512, False), (2048, 2048, 2048, 8200, False), (4096, 4096, 4096, 4096, False)])
def test_where_last_linears_take_large_tiles(m, n, k1, k2, large):
    from kestrel_amd.ops import fast

    code = fast.pair_large_parts(m, n, k1, k2)
    assert (code > 0) == large
    if large:
        bf = dict(dtype=torch.bfloat16, device=DEV)
        args = (torch.zeros(m, k1, **bf), torch.zeros(n, k1, **bf), None, torch.zeros(m, k2, **bf), torch.zeros(n, k2, **bf), None, torch.zeros(m, n, device=DEV))
        assert not fast.linear_pair_accumulate(*args) and fast.linear_pair_accumulate(*args, large=True)
