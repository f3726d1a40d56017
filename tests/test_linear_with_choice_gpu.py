"""A router's choice beside a linear in its launch: the bits of the two launches."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("m", [1, 2, 7, 8])
# (widths of 1, 2, 4, 5, 6 and 8 pieces a wave, some with a last one that is not whole; outputs of whole strips and not)
@pytest.mark.parametrize("k, outputs, extra, n", [(64, 4, 0, 8), (520, 30, 2, 64), (1032, 64, 0, 12), (2048, 32, 0, 2048), (2560, 33, 3, 2560), (2816, 30, 2, 2048), (4096, 12, 0, 516)])
def test_choice_in_a_linears_launch(m, k, outputs, extra, n):
    from kestrel_amd.ops import core, fast

    gen = torch.Generator().manual_seed(m + k + outputs)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    a, w = rnd(m, k).bfloat16().to(DEV), (rnd(n, k) * k ** -0.5).bfloat16().to(DEV)
    rows = w.shape[0]
    bias = rnd(rows).to(DEV) if rows % 4 == 0 else None
    given = rnd(m, outputs + extra).to(DEV)
    correction = (rnd(outputs) * 0.1).to(DEV)
    for options in (dict(), dict(scores="sigmoid", always=outputs), dict(weigh_chosen=True)):
        groups, keep = (2, 1) if outputs % 2 == 0 and not options.get("weigh_chosen") else (0, 0)
        top = min(4, outputs // 2)
        fix = None if options.get("weigh_chosen") else correction
        results = []
        for fused in (True, False):
            out = torch.full((m, rows), float("nan"), device=DEV)
            chosen = torch.full((m, top + ("always" in options)), -7, dtype=torch.int32, device=DEV)
            weights = torch.full(chosen.shape, float("nan"), device=DEV)
            choice = (given, outputs, fix, top, groups, keep, 1.5, chosen, weights)
            if fused:
                assert fast.linear_choice(a, w, bias, out, *choice, **options)
            else:
                assert fast.linear_bf16(a, w, bias, out, 0, False)
                core.route(*choice, **options)
            results.append([t.cpu() for t in (out, chosen, weights)])
        assert all(torch.equal(x, y) for x, y in zip(*results))
        assert torch.isfinite(results[0][0]).all() and int(results[0][1].min()) >= 0


def test_what_is_not_covered_runs_nothing():
    from kestrel_amd.ops import fast

    def call(m, k, outputs, n):
        out, logits = torch.full((m, n), 3.0, device=DEV), torch.zeros(m, outputs, device=DEV)
        chosen, weights = torch.full((m, 2), -7, dtype=torch.int32, device=DEV), torch.zeros(m, 2, device=DEV)
        done = fast.linear_choice(torch.ones(m, k, device=DEV, dtype=torch.bfloat16), torch.ones(n, k, device=DEV, dtype=torch.bfloat16), None, out,
                                  logits, outputs, None, 2, 0, 0, 1.0, chosen, weights)
        assert done or (bool((out == 3.0).all()) and bool((chosen == -7).all()))
        return done

    assert call(8, 256, 64, 64) and not call(9, 256, 64, 64) and not call(8, 256, 65, 64)
    assert call(1, 4096, 8, 64) and not call(1, 4104, 8, 64)   # (rows too long for the kernel's registers)
