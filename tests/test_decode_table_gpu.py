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
