"""Decode attention by the width of the block table: up to 2,048 pages a row's table is always read from LDS, beyond it is where it fits there."""

from __future__ import annotations

import pytest
import torch

from tests.test_kernels_gpu import DEV, PagedCase, _close, _run_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", [4, 8, 16])
@pytest.mark.parametrize("hd", [16, 64, 80, 128])
def test_a_wider_table_changes_nothing(hd, waves, monkeypatch):
    """The same rows behind tables of their own width, of 2,048 and of 2,049 entries: the same bits."""
    from kestrel_amd.ops import fast

    shape_of = fast.decode_shape
    monkeypatch.setattr(fast, "decode_shape", lambda max_kv, workgroups=1, head_dim=64: (shape_of(max_kv, workgroups, head_dim)[0], waves))
    case = PagedCase([1000, 1, 64, 17], [1] * 4, 4, 2, hd, 16, torch.bfloat16, seed=hd + waves)
    narrow = _run_attention(case, "fast", hd ** -0.5)
    _close(narrow, case.reference(hd ** -0.5), torch.bfloat16)
    rows = case.table
    for width in (2048, 2049):
        case.table = torch.zeros(rows.shape[0], width, dtype=torch.int32, device=DEV)
        case.table[:, :rows.shape[1]] = rows
        assert torch.equal(_run_attention(case, "fast", hd ** -0.5), narrow)


@pytest.mark.parametrize("keys", [32768, 32769])
@pytest.mark.parametrize("hd", [64, 80])
def test_rows_at_the_edge_of_the_table_in_lds(hd, keys):
    case = PagedCase([keys, 33], [1, 1], 1, 1, hd, 16, torch.bfloat16, seed=hd)
    _close(_run_attention(case, "fast", hd ** -0.5), case.reference(hd ** -0.5), torch.bfloat16)


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("hd", [64, 80])
@pytest.mark.parametrize("width", [2, 4])
def test_a_row_longer_than_its_table_reads_what_the_table_holds(hd, waves, width, monkeypatch):
    """Keys without an entry weigh nothing; rows that fit are as they were. The token's own key, where the kernel rotates and stores it, counts either way."""
    from kestrel_amd.ops import fast

    shape_of = fast.decode_shape
    monkeypatch.setattr(fast, "decode_shape", lambda max_kv, workgroups=1, head_dim=64: (shape_of(max_kv, workgroups, head_dim)[0], waves))
    case = PagedCase([200, 33, 32, 1], [1] * 4, 4, 2, hd, 16, torch.bfloat16, seed=hd + waves)
    case.table = case.table[:, :width].contiguous()
    rows, lo, hi = case.lists
    case.lists = (rows, lo, [min(k, width * 16) for k in hi])
    _close(_run_attention(case, "fast", hd ** -0.5), case.reference(hd ** -0.5), torch.bfloat16)
    # fused: the same caches, one more key that is the token's own
    gen = torch.Generator().manual_seed(hd)
    qkv = torch.randn(4, 8 * hd, generator=gen).bfloat16().to(DEV)
    angles = torch.zeros(256, 16, device=DEV)
    angles[:, :8] = 1.0                                          # (cosines, then sines: no rotation)
    out, longer = torch.full((4, 4 * hd), float("nan"), dtype=torch.bfloat16, device=DEV), case.kv_hi + 1
    slots = torch.full((4,), -1, dtype=torch.int32, device=DEV)
    assert fast.attention_decode_bf16(qkv, case.k_cache, case.v_cache, case.table, case.token_row, None, longer, out, hd ** -0.5, 4, 2, hd, case.batch,
                                      fuse=(qkv[:, 4 * hd:6 * hd], qkv[:, 6 * hd:], angles, slots))
    q, k_new, v_new = (t.cpu().double() for t in (qkv[:, :4 * hd].view(4, 4, hd), qkv[:, 4 * hd:6 * hd].view(4, 2, hd), qkv[:, 6 * hd:].view(4, 2, hd)))
    want = torch.empty(4, 4, hd, dtype=torch.float64)
    for t, end in enumerate(case.lists[2]):
        for head in range(4):
            keys = torch.cat([case.k[t][:end, head // 2].double(), k_new[t, head // 2][None]])
            values = torch.cat([case.v[t][:end, head // 2].double(), v_new[t, head // 2][None]])
            want[t, head] = torch.softmax(keys @ q[t, head] * hd ** -0.5, dim=0) @ values
    _close(out, want.view(4, -1), torch.bfloat16)


# K of the linear beside it: one, two and four blocks of 64 a wave
@pytest.mark.parametrize("h, hkv, hd, k", [(4, 4, 64, 512), (6, 2, 48, 520), (2, 1, 16, 1024), (32, 32, 64, 2048)])
def test_a_wider_table_changes_nothing_beside_a_linear(h, hkv, hd, k):
    """The launch with a linear layer on the side, rows behind tables of their own width, of 2,048 and of 2,049 entries: the same bits of both."""
    from kestrel_amd.ops import fast
    from kestrel_amd.parts import SideLinear

    gen = torch.Generator().manual_seed(hd + k)
    lens = [1000, 33, 64][:max(1, 128 // h)]
    case = PagedCase(lens, [1] * len(lens), h, hkv, hd, 16, torch.bfloat16, seed=hd)
    n = len(lens)
    a, w = (torch.randn(rows, k, generator=gen).bfloat16().to(DEV) for rows in (n, 520))
    q, rows = case.q.to(DEV), case.table
    results = []
    for width in (rows.shape[1], 2048, 2049):
        table = torch.zeros(rows.shape[0], width, dtype=torch.int32, device=DEV)
        table[:, :rows.shape[1]] = rows
        out, linear = torch.full((n, h * hd), float("nan"), dtype=torch.bfloat16, device=DEV), torch.full((n, 520), float("nan"), device=DEV)
        job = SideLinear(a, w, None, linear, 0)
        assert fast.attention_decode_takes(job, n, h, hd, 16, case.batch.max_kv)
        assert fast.attention_decode_bf16(q, case.k_cache, case.v_cache, table, case.token_row, None, case.kv_hi, out, hd ** -0.5, h, hkv, hd, case.batch, beside=job)
        results.append((out, linear))
    _close(results[0][0], case.reference(hd ** -0.5), torch.bfloat16)
    want = a.double() @ w.double().T
    assert bool(((results[0][1].double() - want).abs() <= (k + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)).all())
    for out, linear in results[1:]:
        assert torch.equal(out, results[0][0]) and torch.equal(linear, results[0][1])
