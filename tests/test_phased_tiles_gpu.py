"""Linears of prompts on the phased tiles: two first linears in one launch, two last ones with K of both in parts, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _rnd(seed):
    gen = torch.Generator().manual_seed(seed)
    return lambda *shape: torch.randn(*shape, generator=gen)


def _close(got, want, magnitudes, count, rounded):
    """A sum of ``count`` products that are exact in 32 bits, in any order, is off by at most count 2^-24 of the sum of magnitudes; rounding it to
    bf16 adds half a step of 8 bits; an activation of slope at most 1.13 passes both on and adds a few steps of 24 bits of its input."""
    bound = 1.13 * (count + 8) * 2.0 ** -24 * magnitudes + (2.0 ** -8 * want.abs() if rounded else 0.0)
    assert bool(((got.double().cpu() - want).abs() <= bound + 2.0 ** -60).all())


# every tile: two K-steps (none in the loop's middle), odd and even numbers of them, rows and columns at the edges of tiles and of their halves
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("m, n1, n2, k", [(65, 8, 264, 128), (257, 520, 136, 192), (128, 256, 128, 320), (383, 192, 1000, 256)])
def test_two_first_linears_in_one_launch(tile, m, n1, n2, k):
    from kestrel_amd.ops import fast

    rnd = _rnd(m + n1 + k)
    a, w1, w2, b1 = rnd(m, k + 8).bfloat16(), rnd(n1, k).bfloat16(), rnd(n2, k + 16).bfloat16(), rnd(n1)
    o1, o2 = (torch.full((m, n + 8), 7.0, dtype=torch.bfloat16, device=DEV) for n in (n1, n2))
    da, dw1, dw2, db1 = (t.to(DEV) for t in (a, w1, w2, b1))
    for act in (1, 3):
        fast._check(fast.lib().ka_linear_joint_bf16(
            da.data_ptr(), k + 8, m, k, dw1.data_ptr(), k, db1.data_ptr(), o1.data_ptr(), n1 + 8, n1, 0,
            dw2.data_ptr(), k + 16, None, o2.data_ptr(), n2 + 8, n2, act, tile, torch.cuda.current_stream().cuda_stream))
        x, y = a[:, :k].double(), w2[:, :k].double()
        _close(o1[:, :n1], x @ w1.double().T + b1.double(), x.abs() @ w1.double().abs().T + b1.double().abs(), k + 1, True)
        z = x @ y.T
        want = torch.nn.functional.gelu(z, approximate="tanh") if act == 1 else torch.nn.functional.silu(z)
        _close(o2[:, :n2], want, x.abs() @ y.abs().T, k, True)
        assert bool((o1[:, n1:] == 7.0).all()) and bool((o2[:, n2:] == 7.0).all())


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
    _close(out, p @ q.T + r @ s.T + rest, p.abs() @ q.abs().T + r.abs() @ s.abs().T + b1.double().abs() + b2.double().abs() + x.double().abs(), k1 + k2 + 3, False)


@pytest.mark.parametrize("m, n1, n2, k, tile", [(64, 6144, 8192, 2048, 0), (65, 6144, 8192, 2048, 6), (257, 6144, 8192, 2048, 3), (513, 6144, 8192, 2048, 2),
                                                (1024, 6144, 8192, 2048, 1), (1025, 6144, 8192, 2048, 0), (257, 6144, 16384, 4096, 0), (300, 6144, 8192, 2056, 0),
                                                (300, 6148, 8192, 2048, 0), (300, 264, 8192, 64, 0)])
def test_where_first_linears_are_one_launch(m, n1, n2, k, tile):
    from kestrel_amd.ops import fast

    assert fast.joint_tile(m, n1, n2, k) == tile


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


@pytest.mark.parametrize("m, large", [(768, False), (1536, True)])
def test_rows_over_more_than_4_gb(m, large):
    """A view whose offsets pass 32 bits of bytes goes where it went without phased tiles: by the small ones, or to the caller's other way."""
    from kestrel_amd.ops import fast

    n, k1, k2 = 2048, 2048, 8192
    rnd = _rnd(m)
    rows = [rnd(m, k).bfloat16().to(DEV) for k in (k1, k2)]
    weights = [(rnd(n, k) * k ** -0.5).bfloat16().to(DEV) for k in (k1, k2)]
    stride = (1 << 31) // (m - 1) // 8 * 8 + 8
    wide = torch.empty(m * stride, dtype=torch.bfloat16, device=DEV).as_strided((m, k2), (stride, 1))
    wide.copy_(rows[1])
    assert (m - 1) * stride + k2 >= 1 << 31
    assert (fast.pair_large_parts(m, n, k1, k2) if large else fast.pair_tile_parts(m, n, k1, k2)) >= fast.PAIR_TILE_CODE
    out = torch.zeros(m, n, device=DEV)
    done = fast.linear_pair_accumulate(rows[0], weights[0], None, wide, weights[1], None, out, large=large)
    assert done == (not large)
    if done:
        x = [t.double().cpu() for t in (*rows, *weights)]
        _close(out, x[0] @ x[2].T + x[1] @ x[3].T, x[0].abs() @ x[2].abs().T + x[1].abs() @ x[3].abs().T, k1 + k2, False)
    else:
        assert bool((out == 0.0).all())


def test_a_replayed_graph_repeats_the_eager_bits():
    from kestrel_amd.ops import fast

    torch.manual_seed(5)
    bf = dict(dtype=torch.bfloat16, device=DEV)
    a, w1, w2, v1, v2 = (torch.randn(*s, **bf) for s in ((520, 512), (1024, 512), (2048, 512), (512, 1024), (512, 2048)))
    fields = [(torch.empty(520, 1024, **bf), torch.empty(520, 2048, **bf), torch.empty(520, 512, device=DEV)) for _ in range(2)]

    def run(o1, o2, x):
        assert fast.linear_joint(a, w1, None, o1, 0, w2, None, o2, 1)
        assert fast.linear_pair_accumulate(o1, v1, None, o2, v2, None, x, accumulate=False)

    run(*fields[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(*fields[1])
    for _ in range(3):
        for t in fields[1]:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(*fields))
        run(*fields[0])


# the tiles of four waves: a part of two K-steps (less than their stages), an odd number, more than the stages, parts of one linear alone, ragged rows and columns
@pytest.mark.parametrize("tile", [5, 8, 10, 12])
@pytest.mark.parametrize("m, n, k1, k2, parts", [(65, 132, 64, 64, 1), (257, 260, 192, 1024, 3), (300, 516, 512, 512, 2), (513, 128, 640, 320, 7), (256, 256, 1088, 64, 2)])
def test_two_last_linears_by_four_waves(tile, m, n, k1, k2, parts):
    test_two_last_linears_in_parts(tile, m, n, k1, k2, parts)
