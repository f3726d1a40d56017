"""Which blocks' two last linears go by tiles: at the lines of the rule."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


# (up to 32 tiles; up to 80 with a long K; up to 128 only in front of a norm; to 160 in front of one in several parts; beyond; few rows)
@pytest.mark.parametrize("m, n, k1, k2, normed, alone", [
    (256, 2048, 512, 512, True, True), (257, 2048, 512, 512, True, False), (512, 2048, 2048, 2048, True, False), (512, 2560, 2560, 10240, True, True),
    (512, 2560, 2560, 2560, True, False), (641, 2048, 2048, 8192, True, False), (1024, 2048, 2048, 2048, True, False), (1025, 2048, 2048, 2048, False, False),
    (1280, 2048, 2048, 8192, True, False), (1281, 2048, 2048, 8192, False, False), (64, 2048, 2048, 8192, False, False), (65, 2048, 2048, 8200, False, False)])
def test_where_pairs_go_by_tiles(m, n, k1, k2, normed, alone, monkeypatch):
    """The rule, and that a block of two branches asks it: its linears are two where it says no."""
    from types import SimpleNamespace

    from kestrel_amd.ops import fast
    from kestrel_amd.ops import linear as linears
    from kestrel_amd.parts import block

    assert fast.pair_tiles_pay(m, n, k1, k2, True) == normed and fast.pair_tiles_pay(m, n, k1, k2, False) == alone
    seen = []
    monkeypatch.setattr(linears, "linear", lambda *a, **k: seen.append("one"))
    monkeypatch.setattr(fast, "linear_pair_accumulate", lambda *a, **k: seen.append("pair") or True)
    weight = lambda k: SimpleNamespace(shape=(n, k))  # noqa: E731
    part = lambda k: SimpleNamespace(input_projection=lambda: (None, None, k, 0), output_projection=lambda: (weight(k), None),  # noqa: E731
                                     attend=lambda *a: None)
    two = SimpleNamespace(mixer=part(k1), feed_forward=part(k2), dtype=torch.bfloat16)
    batch = SimpleNamespace(workspace=SimpleNamespace(get=lambda *a: None))
    rows = SimpleNamespace(shape=(m, n))
    assert block._two_branches_by_stages(two, rows, rows, batch, None, rows)
    assert seen == ["one", "one"] + (["pair"] if alone or m <= fast.SKINNY_MAX_ROWS else ["one", "one"])


# (129 to 160 tiles: with K in parts they pay whatever tile is chosen, its borders are no borders of the rule)
@pytest.mark.parametrize("n, k1, k2, pays", [(2048, 2048, 8192, True), (2048, 1024, 5888, True), (2048, 2048, 4096, True), (2560, 2560, 10240, True),
                                             (1536, 1536, 6144, True), (4096, 4096, 8192, True), (1024, 1024, 4992, True), (2048, 2048, 2048, False),
                                             (2560, 512, 2560, False)])
def test_pairs_in_parts_pay_up_to_160_tiles_of_any_kind(n, k1, k2, pays):
    from kestrel_amd.ops import fast

    across = -(-n // 128)
    rows = range(128 // across * 128 + 1, 160 // across * 128 + 1, 13)
    tiles = {fast.pair_tile_parts(m, n, k1, k2) // fast.PAIR_TILE_CODE for m in rows}
    assert [fast.pair_tiles_pay(m, n, k1, k2, True) for m in rows] == [pays] * len(rows)
    assert not pays or tiles & {1, 3}
