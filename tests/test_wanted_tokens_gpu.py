"""The last layer for the wanted tokens alone, against the same steps with all tokens of it, and the kernel that picks rows out."""

import pytest
import torch

from tests import bogivik_cases, bokorax_cases, gozatar_cases, helpers, vufolorn_cases
from tests.plain import moondream_plain as plain

pytestmark = pytest.mark.gpu

CASES = [("moondream2", "C"), ("moondream2", "F")] + \
    [(family, name) for family in ("bogivik", "bokorax", "gozatar", "vufolorn") for name in "PQRS"]
FOLDERS = {"bogivik": lambda name, dtype: bogivik_cases.model_dir(name), "bokorax": bokorax_cases.folder_for, "gozatar": gozatar_cases.folder_for, "vufolorn": vufolorn_cases.folder_for}

# (request, tokens, wanted places) of every step: nothing wanted; the last places of portions, several of one and places inside; a decoded token
# beside portions, more of them wanted than half (all tokens of the last layer, also without the rule); portions of 70 and 81 tokens, so
# that graphs of 64 and more tokens and the eager path both come; decoded tokens that read what those steps have left
STEPS = [
    [("a", 40, ())],
    [("a", 30, (29,)), ("b", 45, (3, 20, 44)), ("c", 20, ())],
    [("a", 1, (0,)), ("b", 1, (0,)), ("c", 37, (36,))],
    [("a", 1, (0,)), ("c", 2, (0, 1))],
    [("a", 70, (69,)), ("b", 81, (80,)), ("c", 3, (2,))],
    [("a", 1, (0,)), ("b", 1, (0,)), ("c", 1, (0,))],
]


def _logits(folder, dtype, graphs):
    from kestrel_amd.engine.loading import load_model, make_runner
    from kestrel_amd.engine.step import StepEntry

    runner = make_runner(load_model(folder, dtype, torch.device("cuda:0")), 16, 64, 4, enable_graphs=graphs)
    helpers.poison_cache(runner)
    slots = {name: runner.admit() for name in "abc"}
    ids = {name: helpers.random_ids(i, 200, runner.model.plan.vocab_size) for i, name in enumerate("abc")}
    at, out = dict.fromkeys("abc", 0), []
    for step in STEPS:
        entries = []
        for name, count, want in step:
            entries.append(StepEntry(slots[name], ids[name][at[name]:at[name] + count], want=want))
            at[name] += count
        out.append(runner.step(entries).clone())
    return torch.cat(out)


@pytest.mark.parametrize("graphs", [False, True], ids=["eager", "graphs"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("family,name", CASES, ids=lambda v: str(v))
def test_last_layer_for_wanted_tokens(monkeypatch, family, name, dtype, graphs):
    from kestrel_amd.engine.batch import WantedTokens

    folder = FOLDERS[family](name, dtype) if family in FOLDERS else helpers.model_dir(name)
    narrow = _logits(folder, dtype, graphs)
    monkeypatch.setattr(WantedTokens, "MOST", -1)
    whole = _logits(folder, dtype, graphs)
    assert narrow.shape == whole.shape and bool(torch.isfinite(whole).all())
    # each side is off from exact numbers by what ``helpers.tolerance`` states at most (for fp32 as a share of a row's spread, for weights of any scale)
    atol, rtol, spread = helpers.tolerance(dtype)
    bound = atol + rtol * whole.abs() + (spread or 2e-5) * whole.std(dim=1, keepdim=True)
    assert bool(((narrow - whole).abs() <= 2 * bound).all()), f"off by {float(((narrow - whole).abs() / bound).max()):.3g} bounds"


@pytest.mark.parametrize("graphs", [False, True], ids=["eager", "graphs"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", ["C", "D", "E", "F"])
def test_wanted_tokens_inside_a_block_that_sees_both_ways(name, dtype, graphs):
    """Given embeddings in front: wanted tokens of them, which see keys behind their own, and of the text, alone and beside a request without any."""
    from kestrel_amd.engine.loading import load_model, make_runner
    from kestrel_amd.engine.step import StepEntry

    cfg = helpers.flat_config(name)
    runner = make_runner(load_model(helpers.model_dir(name), dtype, torch.device("cuda:0")), 16, 64, 4, enable_graphs=graphs)
    helpers.poison_cache(runner)
    weights = helpers.stored_weights(helpers.model_dir(name))
    prefix = torch.randn(37, cfg["dim"], generator=torch.Generator().manual_seed(9))
    ids = {tag: helpers.random_ids(i, 60, cfg["vocab_size"]) for i, tag in enumerate("ab")}
    first, second = runner.admit(), runner.admit()
    embeds = prefix.to("cuda:0")
    inside = StepEntry(first, [-1] * 37 + ids["a"][:20], want=(0, 18, 36, 50), embeds=embeds, bidirectional=[(0, 37)])
    steps = [[StepEntry(second, ids["b"][:25], want=(24,)), inside], [StepEntry(second, ids["b"][25:55], want=(3, 29)), StepEntry(first, ids["a"][20:30], want=(9,))]]
    places = [[("b", 24), ("a", 0), ("a", 18), ("a", 36), ("a", 50)], [("b", 28), ("b", 54), ("a", 66)]]
    want = {"a": plain.forward(cfg, weights, ids["a"][:30], prefix), "b": plain.forward(cfg, weights, ids["b"][:55], None)}
    for entries, order in zip(steps, places):
        logits = runner.step(entries)
        helpers.assert_close(logits, torch.stack([want[tag][place] for tag, place in order]), dtype, f"tiny {name}")


@pytest.mark.parametrize("m", [0, 1, 7, 64])
def test_gather_rows(m):
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(m)
    rows = torch.randint(0, 90, (m,), generator=gen).to("cuda:0", torch.int32)
    wide = torch.randn(90, 301, device="cuda:0")
    sources = [wide[:, :256], wide[:, 1:30], torch.randn(90, 4, 100, device="cuda:0"), torch.randn(90, 515, device="cuda:0").bfloat16()[:, 1:514],
               torch.arange(90, dtype=torch.int32, device="cuda:0")] * 3          # (more than one launch)
    outs = [torch.full((m, *s.shape[1:]), 7, dtype=s.dtype, device="cuda:0") for s in sources]
    outs[0] = torch.full((m, 300), 7.0, device="cuda:0")[:, 4:260]
    core.gather_rows(rows, list(zip(sources, outs)))
    for source, out in zip(sources, outs):
        assert torch.equal(out, source[rows.long()])
    with pytest.raises(core.KernelError):
        core.gather_rows(rows, [(wide[:, :256], outs[1])])
