"""Sums whose order is the same whatever tile, number of threads or kernel a step's size calls for: equal bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("n, dim, ff", [(1, 80, 16), (150, 208, 80), (257, 144, 336)])
def test_listed_experts_do_not_depend_on_the_tile(n, dim, ff, gated):
    """The kernel for sizes in no steps of 64 and the tiles for those that are, the same operands with zeros behind their last channel."""
    from kestrel_amd.engine.batch import Workspace
    from kestrel_amd.ops import fast
    from kestrel_amd.ops.linear import ACT_GATED, activation_code

    gen = torch.Generator().manual_seed(n + dim + ff)
    n_experts, top = 5, 3
    act = activation_code("silu") | ACT_GATED if gated else activation_code("relu_squared")
    h = torch.randn(n, dim, generator=gen).bfloat16()
    first = (torch.randn(n_experts, ff * (2 if gated else 1), dim, generator=gen) * dim ** -0.5).bfloat16()
    down = (torch.randn(n_experts, dim, ff, generator=gen) * ff ** -0.5).bfloat16()
    chosen = torch.stack([torch.randperm(n_experts, generator=gen)[:top] for _ in range(n)]).to(torch.int32).to(DEV)
    dim64, ff64 = -(-dim // 64) * 64, -(-ff // 64) * 64
    assert dim64 > dim and ff64 > ff
    pad = lambda t, *sizes: torch.nn.functional.pad(t, [x for have, want in zip(reversed(t.shape), reversed(sizes)) for x in (0, want - have)])  # noqa: E731
    results = []
    for operands, width, tiles in (((h, first, down), dim, (128,)),
                                   ((pad(h, n, dim64), pad(first, n_experts, first.shape[1] // ff * ff64, dim64), pad(down, n_experts, dim64, ff64)), dim64,
                                    (64, 128, 256))):
        for tile in tiles:
            y = torch.full((n * top, width), float("nan"), device=DEV)
            assert fast.experts_feed_forward_bf16(*(t.to(DEV) for t in operands), chosen, None, y, act, Workspace(torch.device(DEV)), tile=tile)
            results.append(y[:, :dim].cpu())
    assert all(torch.equal(results[0], other) for other in results[1:])


@pytest.mark.parametrize("dim", [1028, 2048, 2560, 4096, 5000, 8192])
def test_rows_of_the_stream_do_not_depend_on_their_number(dim):
    """Many rows get 256 threads each, few get one a piece: the numbers of a row are the same bits."""
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(dim)
    n, few, top, E, S = 1100, 5, 4, 6, 4                       # (1,100: more than two rows a CU)
    rnd = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)  # noqa: E731
    streams, x, y, h, shared = rnd(n, S, dim), rnd(n, dim), rnd(n * top, dim), rnd(n, dim).bfloat16(), rnd(n, dim)
    chosen = torch.randint(0, E + 1, (n, top), generator=gen).to(torch.int32).to(DEV)
    weights, mix, out, into, gain, gain2 = rnd(n, top).abs(), rnd(S, S), rnd(S), rnd(S), rnd(dim), rnd(dim)

    def results(m):
        done = []
        for kind in ("layernorm", "rms"):
            got, rows = streams[:m].clone(), torch.full((m, dim), float("nan"), device=DEV)
            core.streams_step(got, x[:m].contiguous(), mix, out, (into, (kind, gain, None, 1e-5)), rows)
            again, left = streams[:m].clone(), torch.full((m, dim), float("nan"), device=DEV)
            core.streams_experts(again, y[:m * top], h[:m].float(), chosen[:m], weights[:m], E, shared[:m], None, mix, out,
                                 (into, (kind, gain, None, 1e-5)), left)
            done += [got, rows, again, left]
        got, rows = x[:m].clone(), torch.full((m, dim), float("nan"), dtype=torch.bfloat16, device=DEV)
        core.experts_combine_normed(y[:m * top], h[:m], chosen[:m], weights[:m], E, shared[:m], None, got, (gain, 1e-5), (gain2, 1e-5), rows)
        again, left = x[:m].clone(), torch.full((m, dim), float("nan"), device=DEV)
        core.add_normed(again, shared[:m].contiguous(), (gain, 1e-5), (gain2, 1e-5), left)
        return [t[:few].cpu() for t in done + [got, rows, again, left]]

    for i, (a, b) in enumerate(zip(results(n), results(few))):
        assert torch.equal(a, b), f"result {i}"


@pytest.mark.parametrize("m", [9, 16, 17, 33, 48, 64])
@pytest.mark.parametrize("n, ks", [(64, (2624,)), (1000, (4096,)), (77, (8192,)), (12288, (2688,)), (640, (64, 320)), (2056, (2048, 8192)), (4096, (192, 64)), (51300, (192,)), (51300, (64, 128))])
def test_few_rows_have_the_bits_of_the_kernel_that_streams_weights(m, n, ks):
    """Tiles for K in steps of 64, and the kernel with activations in LDS: the same parts of K, the same order within."""
    from kestrel_amd.ops import fast

    gen = torch.Generator().manual_seed(m + n + sum(ks))
    rows = [torch.randn(m, k, generator=gen).bfloat16().to(DEV) for k in ks]
    weights = [torch.randn(n, k, generator=gen).bfloat16().to(DEV) for k in ks]
    bias, start = torch.randn(n, generator=gen).to(DEV), torch.randn(m, n, generator=gen).to(DEV)
    results = []
    try:
        for mode in (1, 2):
            fast.set_skinny_wide(mode)
            out = start.clone()
            if len(ks) == 1:
                assert fast.linear_bf16(rows[0], weights[0], bias, out, 0, True)
            else:
                assert fast.linear_pair_accumulate(rows[0], weights[0], bias, rows[1], weights[1], None, out)
            results.append(out)
    finally:
        fast.set_skinny_wide(1)
    if m > 16 or (len(ks) == 2 and fast.pair_finishes_rows(m, n)):         # (else rule and test name two kernels)
        assert torch.equal(*results)
    want = start.double() + bias.double() + sum(a.double() @ w.double().T for a, w in zip(rows, weights))
    assert float((results[0].double() - want).norm() / want.norm()) < 2.0 ** -20


@pytest.mark.parametrize("clamped", [False, True])
@pytest.mark.parametrize("n, top, n_experts, dim, ff", [(1, 1, 1, 64, 64), (33, 4, 30, 448, 704), (128, 4, 30, 2048, 704), (85, 6, 62, 256, 896), (512, 1, 3, 192, 128),
                                                        (40, 6, 5, 320, 64)])
def test_lists_of_few_pairs_have_the_bits_of_the_kernel_of_few(n, top, n_experts, dim, ff, clamped):
    """Up to 512 pairs an expert's weights are streamed past its pairs or its pairs are listed and go by tiles: the same order of every sum."""
    from kestrel_amd.engine.batch import Workspace
    from kestrel_amd.ops import fast
    from kestrel_amd.ops.linear import ACT_GATED, activation_code
    from kestrel_amd.parts.specs import GateClamp

    gen = torch.Generator().manual_seed(n + dim + ff)
    h = torch.randn(n, dim, generator=gen).bfloat16().to(DEV)
    clamp = GateClamp(0.7, 1.702, 1.0) if clamped else None
    chosen = torch.stack([torch.randperm(n_experts + 1, generator=gen)[:top] for _ in range(n)]).to(torch.int32).to(DEV)
    down = (torch.randn(n_experts, dim, ff, generator=gen) * ff ** -0.5).bfloat16().to(DEV)
    for act, rows in ((activation_code("silu") | ACT_GATED, 2 * ff), (activation_code("relu_squared"), ff)):
        if clamped and not act & ACT_GATED:
            continue
        first = (torch.randn(n_experts, rows, dim, generator=gen) * dim ** -0.5).bfloat16().to(DEV)
        few, listed = (torch.full((n * top, dim), 7.0, device=DEV) for _ in range(2))
        assert fast.experts_few_bf16(h, first, down, chosen, torch.empty(n * top, ff, dtype=torch.bfloat16, device=DEV), few, act, clamp=clamp)
        assert fast.experts_feed_forward_bf16(h, first, down, chosen, None, listed, act, Workspace(torch.device(DEV)), clamp=clamp)
        assert torch.equal(few, listed)


@pytest.mark.parametrize("n, k", [(64, 32), (130, 96), (2048, 2048), (514, 100)])
def test_gated_linears_in_32_bits_do_not_depend_on_the_rows_beside(n, k):
    """One to forty rows: the same bits for a row, K in steps of 32 (matrix pipes) or not (both vector kernels)."""
    from kestrel_amd.ops import core
    from kestrel_amd.ops.linear import ACT_GATED, activation_code

    gen = torch.Generator().manual_seed(n + k)
    a, w, bias = (torch.randn(*shape, generator=gen) for shape in ((40, k), (n, k), (n,)))
    act = activation_code("silu") | ACT_GATED
    results = {}
    for m in (40, 33, 17, 16, 9, 1):
        out = torch.full((m, n // 2), float("nan"), device=DEV)
        core.linear_generic(a[:m].to(DEV), w.to(DEV), bias.to(DEV), out, act=act)
        results[m] = out.cpu()
    assert all(torch.equal(got, results[40][:m]) for m, got in results.items())
    z = (a.double() @ w.double().T + bias.double()).view(40, n // 2, 2)
    want = z[..., 0] * torch.sigmoid(z[..., 0]) * z[..., 1]
    assert float((results[40].double() - want).norm() / want.norm()) < 2.0 ** -20


# (of 32 heads 16 tokens are two workgroups a CU of 256, 17 are more)
@pytest.mark.parametrize("hd, hdv, page", [(64, 64, 16), (128, 96, 12), (256, 200, 32)])
@pytest.mark.parametrize("window", [False, True])
def test_attention_in_32_bits_does_not_depend_on_the_tokens_beside(hd, hdv, page, window):
    """A token's keys by one wave or by several: the numbers of a token are the same bits alone and in a step of any size."""
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(hd + window)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    n, heads, kv_heads, longest = 150, 32, 8, 700
    pages = -(-longest // page)
    table = torch.randperm(3 * pages, generator=gen).to(torch.int32).view(3, pages).to(DEV)
    k_cache, v_cache = rnd(3 * pages, kv_heads, page, hd).to(DEV), rnd(3 * pages, kv_heads, hdv, page).to(DEV)
    q, sinks = rnd(n, heads * hd).to(DEV), rnd(heads).to(DEV)
    hi = torch.randint(1, longest + 1, (n,), generator=gen).to(torch.int32)
    hi[:4] = torch.tensor([longest, 1, 64, 65])
    row = torch.arange(n, dtype=torch.int32) % 3
    lo = (hi - 300).clamp(min=0).to(DEV) if window else None
    options = dict(value_dim=hdv, keep_first=5, sinks=sinks) if window else dict(value_dim=hdv)
    hi, row = hi.to(DEV), row.to(DEV)

    def results(a, b):
        out = torch.full((b - a, heads * hdv), float("nan"), device=DEV)
        core.attention_generic(q[a:b], k_cache, v_cache, table, row[a:b], lo[a:b] if window else None, hi[a:b], out, hd ** -0.5, heads, kv_heads, hd, **options)
        return out

    whole = results(0, n)
    assert bool(torch.isfinite(whole).all())
    for size in (1, 3, 16, 17, 75):
        assert torch.equal(torch.cat([results(a, min(n, a + size)) for a in range(0, n, size)]), whole), f"steps of {size}"
