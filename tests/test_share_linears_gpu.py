"""Linears of at most eight rows whose workgroups ask for their whole share of the weights at once (``csrc/ka_share.h``), at the edges of its forms:
strips that do not divide over the workgroups, a last strip that is not whole, K in no steps of 64, one strip of a long K, two segments, the norm in front."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
GELU = 1


def _rows(gen, m, k, scale=1.0):
    return (torch.randn(m, k, generator=gen) * scale).bfloat16()


def _sum_slack(a, w, k, more=0.0):
    """A sum of K products in fp32 is off by at most (K + 4) 2^-24 of their magnitudes."""
    return ((k + 4) * 2.0 ** -24 + more) * (a.double().abs() @ w.double().abs().T)


# strips (N / 8) of 256 CUs: under one each, just one, two to nine with a remainder; K: one to eight blocks a wave, then 9 to 26 for one strip
@pytest.mark.parametrize("m", [1, 3, 8])
@pytest.mark.parametrize("n, k", [(4, 8), (12, 520), (2048, 2048), (2056, 1000), (4100, 1544), (6148, 2048), (9280, 2048), (18432, 2056), (12292, 3080), (10240, 4096),
                                  (2048, 4616), (1000, 8448), (2044, 10752), (4096, 13304), (4092, 5000)])
def test_one_linear(m, n, k):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + n + k)
    a, w, bias = _rows(gen, m, k), _rows(gen, n, k, k ** -0.5), torch.randn(n, generator=gen)
    want, slack = a.double() @ w.double().T, _sum_slack(a, w, k)
    out = torch.full((m, n), float("nan"), device=DEV)
    assert fast.linear_bf16(a.to(DEV), w.to(DEV), bias.to(DEV), out, 0, False)
    assert bool(((out.cpu().double() - want - bias.double()).abs() <= slack + 2.0 ** -23 * (want + bias.double()).abs() + 1e-30).all())
    start = torch.randn(m, n, generator=gen)
    out = start.to(DEV)
    assert fast.linear_bf16(a.to(DEV), w.to(DEV), None, out, 0, True)
    assert bool(((out.cpu().double() - want - start.double()).abs() <= slack + 2.0 ** -23 * (want + start.double()).abs() + 1e-30).all())


@pytest.mark.parametrize("m", [1, 5, 8])
@pytest.mark.parametrize("na, nb, k", [(40, 36, 1024), (6144, 8192, 2048), (2052, 4096, 1096), (7680, 10240, 2560)])
def test_two_linears_of_the_same_rows(m, na, nb, k):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + na + k)
    a, wa, wb = _rows(gen, m, k), _rows(gen, na, k, k ** -0.5), _rows(gen, nb, k, k ** -0.5)
    outs = [torch.full((m, n), float("nan"), device=DEV) for n in (na, nb)]
    assert fast.linear_two_outputs(a.to(DEV), wa.to(DEV), None, outs[0], 0, wb.to(DEV), None, outs[1], 0)
    for w, out in zip((wa, wb), outs):
        assert bool(((out.cpu().double() - a.double() @ w.double().T).abs() <= _sum_slack(a, w, k) + 1e-30).all())


@pytest.mark.parametrize("m", [1, 4, 8])
@pytest.mark.parametrize("n, k1, k2", [(2048, 2048, 8192), (2560, 2560, 10240), (72, 2104, 2504), (2052, 64, 4608)])
def test_two_segments(m, n, k1, k2):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + n + k1)
    a, w = [_rows(gen, m, k) for k in (k1, k2)], [_rows(gen, n, k, k ** -0.5) for k in (k1, k2)]
    biases, start = torch.randn(2, n, generator=gen), torch.randn(m, n, generator=gen)
    out = start.to(DEV)
    assert fast.linear_pair_accumulate(a[0].to(DEV), w[0].to(DEV), biases[0].to(DEV), a[1].to(DEV), w[1].to(DEV), biases[1].to(DEV), out)
    sums = [x.double() @ y.double().T for x, y in zip(a, w)]
    want = sums[0] + sums[1] + biases.double().sum(dim=0) + start.double()
    slack = _sum_slack(a[0], w[0], k1 + k2) + _sum_slack(a[1], w[1], k1 + k2) + 3 * 2.0 ** -24 * (biases.abs().sum(dim=0) + start.abs() + want.abs())
    assert bool(((out.cpu().double() - want).abs() <= slack).all())


@pytest.mark.parametrize("m", [1, 4, 5, 8])
@pytest.mark.parametrize("na, nb, k", [(6144, 0, 2048), (6144, 8192, 2048), (7680, 10240, 2560), (24, 2052, 1032), (2052, 0, 2008), (4096, 0, 2056)])
@pytest.mark.parametrize("form", ["shift", "no shift", "uncentred"])
def test_a_norm_in_front(form, m, na, nb, k):
    """Rows far from zero, so that the squares about the mean are not those about zero. The normalised rows are rounded to bf16 (half a unit of the
    last of eight bits: 2^-8) and are off before that by the rounding of the row's sums, some 2^-20 of a standard deviation per unit of mean over deviation."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + na + k)
    x, gamma, beta = torch.randn(m, k, generator=gen) * 3 + torch.arange(m)[:, None] - 2.0, torch.randn(k, generator=gen), torch.randn(k, generator=gen)
    wa, wb = _rows(gen, na, k, k ** -0.5), _rows(gen, max(nb, 4), k, k ** -0.5)
    beta = beta if form == "shift" else None
    xd = x.double()
    centred = xd if form == "uncentred" else xd - xd.mean(dim=1, keepdim=True)
    h = centred / torch.sqrt((centred * centred).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()
    off = 8 * 2.0 ** -20 * gamma.double().abs()
    if beta is not None:
        h = h + beta.double()
    h_slack = 1.01 * 2.0 ** -8 * h.abs() + off
    out_a, out_b = (torch.full((m, n), float("nan"), device=DEV) for n in (na, max(nb, 4)))
    args = (x.to(DEV), gamma.to(DEV), beta.to(DEV) if beta is not None else None, 1e-5, wa.to(DEV), None, out_a, 0)
    stored = None
    if nb:
        assert fast.layernorm_linear(*args, wb.to(DEV), None, out_b, 0, centred=form != "uncentred")
    elif form == "uncentred":
        assert fast.layernorm_linear(*args, centred=False)
    else:
        stored = torch.full((m, k + 8), float("nan"), dtype=torch.bfloat16, device=DEV)[:, :k]
        assert fast.layernorm_linear(*args, store=stored)
        assert bool(((stored.cpu().double() - h).abs() <= h_slack).all())
    for w, out in ((wa, out_a),) + (((wb, out_b),) if nb else ()):
        slack = h_slack @ w.double().abs().T + (k + 4) * 2.0 ** -24 * (h.abs() @ w.double().abs().T)
        assert bool(((out.cpu().double() - h @ w.double().T).abs() <= slack).all())


# outputs of two segments: strips of which a CU holds one or two
@pytest.mark.parametrize("n, k1, k2", [(2048, 2048, 8192), (2560, 2560, 10240), (4096, 4096, 6144), (4096, 2048, 704)])
def test_two_segments_do_not_depend_on_the_rows_beside(n, k1, k2):
    """One row alone, among three and among as many as go this way: the same bits."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(n + k1 + k2)
    a = [_rows(gen, 8, k).to(DEV) for k in (k1, k2)]
    w = [_rows(gen, n, k, k ** -0.5).to(DEV) for k in (k1, k2)]
    start = torch.randn(8, n, generator=gen).to(DEV)
    most = 4 if fast.pair_finishes_rows(8, n) else 8           # (five to eight rows of more strips than CUs: K in parts)
    results = {}
    for m in (most, 3, 1):
        out = start[:m].clone()
        assert fast.linear_pair_accumulate(a[0][:m], w[0], None, a[1][:m], w[1], None, out)
        results[m] = out
    assert torch.equal(results[most][:3], results[3]) and torch.equal(results[most][:1], results[1])


# K: two to five blocks a wave, in steps of 64 and not; outputs: one to seven strips a CU
@pytest.mark.parametrize("n, k", [(2048, 1096), (6144, 1536), (4100, 2008), (14336, 2048), (40, 2048), (6144, 2560), (2052, 2104)])
@pytest.mark.parametrize("form", ["shift", "no shift", "uncentred"])
def test_a_norm_in_front_does_not_depend_on_the_rows_beside(form, n, k):
    """One to sixteen rows, on either side of eight: the same bits of a row, and of what is left of the norm. Rows of one sign, whose sums have to round."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(n + k)
    x = (torch.randn(16, k, generator=gen).abs() * torch.linspace(0.5, 40.0, 16)[:, None]).to(DEV)
    gamma, beta = torch.randn(k, generator=gen).to(DEV), torch.randn(k, generator=gen).to(DEV)
    w = _rows(gen, n, k, k ** -0.5).to(DEV)
    results = {}
    for m in (16, 9, 8, 7, 4, 1):
        out, left = torch.full((m, n), float("nan"), device=DEV), torch.full((m, k), float("nan"), dtype=torch.bfloat16, device=DEV)
        if form == "uncentred":
            assert fast.layernorm_linear(x[:m], gamma, None, 1e-5, w, None, out, 0, centred=False)
            left = None
        else:
            assert fast.layernorm_linear(x[:m], gamma, beta if form == "shift" else None, 1e-5, w, None, out, 0, store=left)
        results[m] = (out, left)
    for m, (out, left) in results.items():
        assert torch.equal(out, results[16][0][:m]), m
        assert left is None or torch.equal(left, results[16][1][:m]), m


# Where the split kernel has nine to sixteen rows: with four waves over K (many strips, or accumulation over a short K), with eight, with eight where it had
# sixteen up to eight rows (few strips)
@pytest.mark.parametrize("n, k, accumulate", [(3288, 4608, False), (4096, 8448, True), (512, 1024, True), (2048, 1280, True), (2048, 1288, True), (2048, 4608, False),
                                              (3272, 8448, True), (256, 8448, False), (1000, 4096, True)])
def test_a_long_or_accumulated_linear_does_not_depend_on_the_rows_beside(n, k, accumulate):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(n + k)
    a, w, start = _rows(gen, 16, k).to(DEV), _rows(gen, n, k, k ** -0.5).to(DEV), torch.randn(16, n, generator=gen).to(DEV)
    results = {}
    for m in (16, 9, 8, 5, 1):
        results[m] = start[:m].clone()
        assert fast.linear_bf16(a[:m], w, None, results[m], 0, accumulate)
    for m, out in results.items():
        assert torch.equal(out, results[16][:m]), m


@pytest.mark.parametrize("m", [1, 5, 8, 12])
@pytest.mark.parametrize("na, nb, k", [(64, 136, 512), (136, 64, 1024), (1000, 1048, 4096)])
def test_accumulation_into_the_first_of_two_targets(m, na, nb, k):
    """The entry point's accumulation is the first target's alone: the second one's outputs are new, also where it is the wider one, and
    its rows lie beside numbers that stay."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + na + k)
    a, wa, wb = _rows(gen, m, k), _rows(gen, na, k, k ** -0.5), _rows(gen, nb, k, k ** -0.5)
    start = torch.randn(m, na, generator=gen)
    ad, wad, wbd, out_a = a.to(DEV), wa.to(DEV), wb.to(DEV), start.to(DEV)
    room = torch.full((m, nb + 8), 7.0, device=DEV)
    out_b = room[:, :nb]
    fast._check(fast.lib().ka_linear_skinny_fused(
        ad.data_ptr(), k, k, None, 0, 0, None, 0, None, None, None, None, 0.0, wad.data_ptr(), k, None, out_a.data_ptr(), 0, na, na, 0, 1,
        wbd.data_ptr(), k, None, out_b.data_ptr(), 0, nb + 8, nb, 0, m, fast.chip_sizes(ad.device).skinny_target_waves, None, 0, fast.stream_ptr()))
    want_a = a.double() @ wa.double().T + start.double()
    assert bool(((out_a.cpu().double() - want_a).abs() <= _sum_slack(a, wa, k) + 2.0 ** -23 * (start.abs() + want_a.abs())).all())
    assert bool(((out_b.cpu().double() - a.double() @ wb.double().T).abs() <= _sum_slack(a, wb, k) + 1e-30).all())
    assert bool((room[:, nb:] == 7.0).all())


# more than nine strips a CU, which the kernel that loops over strips has
@pytest.mark.parametrize("m", [1, 5, 8])
@pytest.mark.parametrize("n, k", [(20484, 520), (20484, 2048), (51200, 1024), (51200, 2048), (18436, 2560), (18436, 4096)])
def test_more_strips_than_a_share(m, n, k):
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + n + k)
    a, w, bias = _rows(gen, m, k).to(DEV), _rows(gen, n, k, k ** -0.5).to(DEV), torch.randn(n, generator=gen).to(DEV)
    out = torch.full((m, n), float("nan"), device=DEV)
    assert fast.linear_bf16(a, w, bias, out, 0, False)
    want = a.double() @ w.double().T + bias.double()
    slack = (k + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T) + 2.0 ** -23 * want.abs()
    assert bool(((out.double() - want).abs() <= slack).all())


@pytest.mark.parametrize("n, k", [(520, 512), (2048, 2048), (4100, 1544), (6148, 2560), (18436, 1024)])
def test_one_linear_does_not_depend_on_the_rows_beside(n, k):
    """Up to 64 rows where the kernel that loops over strips keeps their activations (K up to 2,560): the same bits of a row."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(n + k)
    a, w = _rows(gen, 64, k).to(DEV), _rows(gen, n, k, k ** -0.5).to(DEV)
    results = {}
    for m in (64, 17, 16, 9, 8, 5, 1):
        results[m] = torch.full((m, n), float("nan"), device=DEV)
        assert fast.linear_bf16(a[:m], w, None, results[m], 0, False)
    for m, out in results.items():
        assert torch.equal(out, results[64][:m]), m
