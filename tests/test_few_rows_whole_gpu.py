"""Linears of 17 to 64 rows by tiles that have all of K: the bits of the kernels that stream weights through registers, and the values."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _tile(m, n, k, halves, n2=0):
    """The tile by which a linear goes, in sixteens of weight rows; 0: by the kernels whose bits these are."""
    from kestrel_amd.ops import fast

    return fast.lib().ka_few_rows_whole_tile(m, n, n2, k, int(halves))


def _near(got, want, dtype):
    """fp32: sums of at most 8,192 products in chains of MFMAs, as ``test_few_rows_tiles_gpu.py``; bf16: half a unit in the last place, 2^-9 of the value."""
    limit = 2.0 ** -20 if dtype == torch.float32 else 2.0 ** -8
    assert float((got.double() - want).norm() / want.norm()) < limit


# (rows: a tile of 32 and of 64, full and with one row more than the last wave's; outputs: 1 to 5 sixteens a tile, the last tile full, of four rows, and one
# beside the line to the next; K: one round of the eight sums, and the longest)
@pytest.mark.parametrize("m", [17, 32, 33, 49, 64])
@pytest.mark.parametrize("n, k", [(3072, 512), (4100, 1536), (8196, 2048), (10240, 2560), (12292, 1024), (16384, 1536)])
def test_rows_have_the_bits_of_sixteen_rows_alone(m, n, k):
    from kestrel_amd.ops import fast

    assert _tile(m, n, k, False) == {3072: 1, 4100: 2, 8196: 3, 10240: 3, 12292: 4, 16384: 4}[n]
    gen = torch.Generator().manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=gen).bfloat16().to(DEV), torch.randn(n, k, generator=gen).bfloat16().to(DEV)
    bias = torch.randn(n, generator=gen).to(DEV)
    for b in (bias, None):
        out = torch.full((m + 1, n), 7.0, device=DEV)
        assert fast.linear_bf16(a, w, b, out[:m], 0, False)
        assert bool((out[m] == 7.0).all())
        for lo in range(0, m, 16):
            hi = min(m, lo + 16)
            alone = torch.empty(hi - lo, n, device=DEV)
            assert fast.linear_bf16(a[lo:hi], w, b, alone, 0, False)
            assert torch.equal(out[lo:hi], alone)
        _near(out[:m], a.double() @ w.double().T + (0 if b is None else b.double()), torch.float32)


# (80 weight rows a tile; 49 rows and more go there, and beyond 2,048 of K)
def test_five_sixteens():
    from kestrel_amd.ops import fast

    assert _tile(50, 17924, 2560, False) == 5
    gen = torch.Generator().manual_seed(5)
    a, w = torch.randn(50, 2560, generator=gen).bfloat16().to(DEV), torch.randn(17924, 2560, generator=gen).bfloat16().to(DEV)
    out, alone = torch.empty(50, 17924, device=DEV), torch.empty(16, 17924, device=DEV)
    assert fast.linear_bf16(a, w, None, out, 0, False) and fast.linear_bf16(a[:16], w, None, alone, 0, False)
    assert torch.equal(out[:16], alone)
    _near(out, a.double() @ w.double().T, torch.float32)


@pytest.mark.parametrize("m", [17, 32, 40, 64])
@pytest.mark.parametrize("n, k", [(8196, 64), (10752, 2624), (12292, 3072), (18564, 320), (20484, 2624), (28672, 192), (51204, 128)])
def test_one_part_has_the_bits_of_the_kernel_with_parts(m, n, k):
    """Three to seven sixteens of weight rows a tile; K of fewer steps than there are stages; into the old values, whatever K."""
    from kestrel_amd.ops import fast

    assert _tile(m, n, k, True) == {8196: 3, 10752: 3, 12292: 4, 18564: 5, 20484: 3, 28672: 4, 51204: 7}[n]
    gen = torch.Generator().manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=gen).bfloat16().to(DEV), torch.randn(n, k, generator=gen).bfloat16().to(DEV)
    bias, start = torch.randn(n, generator=gen).to(DEV), torch.randn(m + 1, n, generator=gen).to(DEV)
    results = []
    try:
        for mode in (1, 2):
            fast.set_skinny_wide(mode)
            out = start.clone()
            assert fast.linear_bf16(a, w, bias, out[:m], 0, True)
            assert torch.equal(out[m], start[m])
            results.append(out[:m])
    finally:
        fast.set_skinny_wide(1)
    assert torch.equal(*results)
    _near(results[0], start[:m].double() + bias.double() + a.double() @ w.double().T, torch.float32)


# (outputs too few or too many for one tile a CU, either side of 48 rows; K in no rounds of the eight sums, or in no whole steps; rows that other kernels take)
@pytest.mark.parametrize("m, n, k, halves", [(48, 3068, 2048, False), (48, 16388, 1536, False), (48, 10244, 2048, False), (49, 1020, 512, False), (49, 16388, 2048, False),
                                             (64, 20484, 2560, False), (64, 8192, 2112, False), (64, 8192, 2080, True), (16, 8192, 2048, False), (65, 8192, 2048, False)])
def test_what_other_kernels_take(m, n, k, halves):
    assert _tile(m, n, k, halves) == 0


@pytest.mark.parametrize("m, ns, k", [(20, (2048, 3072), 1024), (64, (6144, 8192), 2048), (40, (8200, 9000), 4096)])
def test_two_outputs_in_bf16(m, ns, k):
    """Two linears of the same rows, the second with an activation, into columns of wider rows; against either alone."""
    from kestrel_amd.ops import fast
    from kestrel_amd.ops.linear import ACT_GATED, activation_code

    assert _tile(m, ns[0], k, k > 2560, ns[1]) == {1024: 2, 2048: 4, 4096: 5}[k]
    gen = torch.Generator().manual_seed(m + sum(ns) + k)
    a = torch.randn(m, k, generator=gen).bfloat16().to(DEV)
    ws = [(torch.randn(n, k, generator=gen) * k ** -0.5).bfloat16().to(DEV) for n in ns]
    bs = [torch.randn(n, generator=gen).to(DEV) for n in ns]
    gelu, gated = activation_code("gelu_tanh"), activation_code("silu") | ACT_GATED
    wide = torch.full((m, sum(ns) + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    outs = [wide[:, :ns[0]], wide[:, ns[0]:ns[0] + ns[1]]]
    assert fast.linear_two_outputs(a, ws[0], bs[0], outs[0], 0, ws[1], bs[1], outs[1], gelu)
    assert bool((wide[:, sum(ns):] == 7.0).all())
    sums = [a.double() @ w.double().T + b.double() for w, b in zip(ws, bs)]
    _near(outs[0], sums[0], torch.bfloat16)
    _near(outs[1], torch.nn.functional.gelu(sums[1], approximate="tanh"), torch.bfloat16)
    for w, b, out, act in zip(ws, bs, outs, (0, gelu)):
        alone = torch.empty(m, w.shape[0], dtype=torch.bfloat16, device=DEV)
        assert fast.linear_bf16(a, w, b, alone, act, False)
        assert torch.equal(alone, out)
    pairs = torch.empty(m, ns[1] // 2, dtype=torch.bfloat16, device=DEV)
    assert fast.linear_bf16(a, ws[1], bs[1], pairs, gated, False)
    _near(pairs, torch.nn.functional.silu(sums[1][:, 0::2]) * sums[1][:, 1::2], torch.bfloat16)
