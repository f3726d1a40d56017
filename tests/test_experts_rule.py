"""Up to how many pairs of a step the chosen experts' weights are streamed past them, by the sizes of a layer of routed experts."""

from __future__ import annotations

import pytest

from kestrel_amd.parts.experts import RoutedExperts
from kestrel_amd.parts.specs import RoutedExpertsSpec


# few experts: 128 pairs would already be many an expert; many: four an expert, to 240; a shared expert among them has a pair of every token; odd sizes
@pytest.mark.parametrize("n_experts, shared, dim, hidden, pairs", [(1, None, 64, 64, 128), (8, None, 4096, 896, 128), (30, None, 2048, 704, 128), (32, None, 2048, 704, 128),
                                                                   (40, None, 2048, 704, 160), (62, None, 4096, 896, 240), (62, 1792, 4096, 896, 240),
                                                                   (256, None, 64, 64, 240), (62, 896, 4096, 896, 128), (62, None, 4096, 880, 512), (8, None, 2040, 64, 512)])
def test_the_line_goes_by_pairs_an_expert(n_experts, shared, dim, hidden, pairs):
    layer = RoutedExperts(RoutedExpertsSpec("routed_experts", dim, n_experts, hidden, 1, shared_hidden=shared, shared_gate=False))
    assert layer.few_pairs_to() == pairs
