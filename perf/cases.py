"""What this engine is timed on: whole requests through ``ModelRunner.step``, from the first prompt portion to the last token.

A case is a batch of requests that arrive together at an engine whose model is loaded and whose graphs are captured. A pass
plans steps as the engine's scheduler does (a token for every request that decodes, the rest of the step's token budget
for prompts, cut where they do not fit; an image is never cut), admits, runs and releases the requests, and leaves the
logits of every sampled place. The tokens that follow a prompt are given with it, so that a rounding cannot send
two implementations along two texts.

Models are those of ``bench.py``: the Moondream 2 text decoder, Phi-2's layer sizes of the same family (heads of 80
channels), and two of the designs with routed experts and a recurrence, Bokorax and Gozatar, at their two benchmark sizes each.
Weights are random N(0, 0.02). The designs with a router get what training gives them and noise does not: token embeddings that
outweigh a single sublayer and that lean towards the experts of the token (with plain noise all tokens of a text would
choose nearly the same experts, by margins of a rounding), and decays over the whole range from fast to slow.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

VOCAB = 51200
PAGE = 16
WEIGHTS_SEED = 2
F64 = torch.float64

# ------------------------------------------------------------------------------------------------ models
_MOONDREAM = {"dim": 2048, "ff_dim": 8192, "n_layers": 24, "vocab_size": VOCAB, "max_context": 2048, "n_heads": 32, "n_kv_heads": 32,
              "rope_theta": 10000.0, "prefix_attn": 730, "layer_norm_eps": 1e-5}
_PHI2 = {"dim": 2560, "ff_dim": 10240, "n_layers": 32, "vocab_size": VOCAB, "max_context": 2048, "n_heads": 32, "n_kv_heads": 32,
         "rope_theta": 10000.0, "prefix_attn": 0, "layer_norm_eps": 1e-5, "rotary_dim": 32}
_BOKORAX = {
    "bokorax-w2048": dict(width=2048, heads=32, kv_heads=8, head=64, window=1024, memory=(32, 64), rank=64,
                          experts=dict(n=30, ff=704, top=4, identity=2, groups=(4, 2), shared=2816), order="2w1s"),
    "bokorax-w4096": dict(width=4096, heads=32, kv_heads=8, head=128, window=2048, memory=(64, 64), rank=128,
                          experts=dict(n=62, ff=896, top=6, identity=2, groups=(8, 4), shared=1792), order="w21"),
}
_GOZATAR = {
    "gozatar-w2048": dict(width=2048, streams=4, heads=32, kv_heads=8, head=64, window=1024, recurrence=(16, 64, 128), rank=64,
                          experts=dict(n=30, ff=704, top=4, groups=(5, 3), shared=704), dense=8448, order="dmmm"),
    "gozatar-w4096": dict(width=4096, streams=4, heads=32, kv_heads=8, head=128, window=2048, recurrence=(32, 64, 128), rank=128,
                          experts=dict(n=62, ff=896, top=6, groups=(2, 1), shared=1792), dense=10752, order="dmm"),
}


def _bokorax_config(s):
    e = s["experts"]
    mlp = {"kind": "moe", "expert": {"ff": e["ff"]}, "shared": {"ff": e["shared"]},
           "router": {"experts": e["n"], "top": e["top"], "identity": e["identity"], "scale": 2.5,
                      "groups": {"count": e["groups"][0], "keep": e["groups"][1]}}}
    common = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["head"], "vdim": s["head"], "scale": s["head"] ** -0.5}
    first = {**common, "mask": {"size": s["window"]}, "rot": {"base": 10000.0, "dims": s["head"] // 2}}
    second = {**common, "softcap": 50.0, "rot": {"base": 500000.0, "dims": s["head"], "scaling": {"factor": 8.0}}}
    memory = {"heads": s["memory"][0], "dim": s["memory"][1], "decay_rank": s["rank"]}
    layers, source = [], None
    for i, kind in enumerate(s["order"]):
        if kind == "w":
            layers.append({"type": "wkv", "mixer": dict(memory), "mlp": mlp})
        elif kind == "1":
            layers.append({"type": "attention", "mixer": dict(first), "mlp": mlp})
        elif kind == "s":
            layers.append({"type": "attention_2", "mixer": dict(second, kv_from=source), "mlp": mlp})
        else:
            layers.append({"type": "attention_2", "mixer": dict(second), "mlp": mlp})
            source = i
    return {"architecture": "Bokorax", "vocab": VOCAB, "width": s["width"], "norm": {"eps": 1e-6}, "embedding": {"scale": 1.0},
            "logit_scale": 1.0, "layers": layers}


def _gozatar_config(s):
    e, (rh, rd, rdv) = s["experts"], s["recurrence"]
    experts = {"kind": "moe", "expert": {"ff": e["ff"], "limit": 7.0}, "shared": {"ff": e["shared"], "limit": 7.0},
               "router": {"experts": e["n"], "top": e["top"], "groups": {"count": e["groups"][0], "keep": e["groups"][1]}}}
    mixer = {"left": {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["head"], "vdim": s["head"], "scale": s["head"] ** -0.5,
                      "conv": 4, "mask": {"size": s["window"]}, "rot": {"base": 10000.0, "dims": s["head"]}},
             "right": {"heads": rh, "dim": rd, "vdim": rdv, "tau": 16.0, "decay_rank": s["rank"]}, "left_scale": 0.8, "right_scale": 1.2}
    layers = [{"type": "parallel", "mixer": mixer, "mlp": {"kind": "dense", "ff": s["dense"]} if kind == "d" else experts} for kind in s["order"]]
    return {"architecture": "Gozatar", "vocab": VOCAB, "width": s["width"], "streams": s["streams"], "norm": {"eps": 1e-5}, "layers": layers}


CONFIGS = {"moondream2": ("moondream2", {"text": _MOONDREAM}), "phi2": ("moondream2", {"text": _PHI2})}
CONFIGS.update({name: ("bokorax", _bokorax_config(s)) for name, s in _BOKORAX.items()})
CONFIGS.update({name: ("gozatar", _gozatar_config(s)) for name, s in _GOZATAR.items()})


# ------------------------------------------------------------------------------------------------ cases
def listed():
    """``rows`` requests, each an image of ``image`` given embeddings (0: none) before ``low`` to ``high`` prompt ids, and ``new`` sampled
    places; ``budget``: the most tokens of a step (2,048 is ``RuntimeConfig``'s default)."""
    return [
        # the smallest call: a short question without an image, a one-word answer; launches and their gaps
        dict(name="short question", model="moondream2", dtype="bf16", rows=1, image=0, low=23, high=23, new=6, budget=2048),
        # one user, one picture: a caption streamed token by token
        dict(name="caption", model="moondream2", dtype="bf16", rows=1, image=730, low=13, high=13, new=40, budget=2048),
        # the longest prompt the model takes (a picture and 1,318 ids), judged by its first token
        dict(name="long prompt", model="moondream2", dtype="bf16", rows=1, image=730, low=1318, high=1318, new=1, budget=2048),
        # eight pictures with questions at once: the benchmark's batch, prompts of about its context
        dict(name="eight pictures", model="moondream2", dtype="bf16", rows=8, image=730, low=37, high=301, new=32, budget=2048),
        # a full batch of short texts
        dict(name="sixty-four texts", model="moondream2", dtype="bf16", rows=64, image=0, low=45, high=333, new=20, budget=2048),
        # continuous batching at Phi-2's sizes: portions of at most 512 tokens beside the decoded tokens of the others
        dict(name="portions", model="phi2", dtype="bf16", rows=10, image=0, low=64, high=1100, new=16, budget=512),
        # the 32-bit path, as trace replays and checks use it
        dict(name="thirty-two bits", model="moondream2", dtype="fp32", rows=3, image=0, low=31, high=157, new=8, budget=2048),
        # texts to be read by a design of attention, a decaying memory and routed experts
        dict(name="reading", model="bokorax-w2048", dtype="bf16", rows=4, image=0, low=700, high=1700, new=2, budget=2048),
        # and a chat of several users with it
        dict(name="chat of eight", model="bokorax-w2048", dtype="bf16", rows=8, image=0, low=90, high=410, new=40, budget=2048),
        # a long document in portions, by the design of several streams at its larger size
        dict(name="document", model="gozatar-w4096", dtype="bf16", rows=1, image=0, low=5300, high=5300, new=2, budget=2048),
        # one user of it at its smaller size
        dict(name="chat of one", model="gozatar-w2048", dtype="bf16", rows=1, image=0, low=201, high=201, new=56, budget=2048),
        # a batch at its larger size
        dict(name="batch of forty", model="gozatar-w4096", dtype="bf16", rows=40, image=0, low=33, high=270, new=24, budget=2048),
    ]


def draw(rng):
    """One more case: any of the models, 1 to 64 requests, prompts of 16 to 2,000 ids, 1 to 48 sampled places, steps of 512 or 2,048
    tokens; no more prompt tokens and no more steps than the largest listed cases have."""
    model = rng.choice(["moondream2", "moondream2", "moondream2", "phi2", *_BOKORAX, *_GOZATAR])
    dtype = "fp32" if model == "moondream2" and rng.random() < 0.2 else "bf16"
    span = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    rows = span(1, 6 if dtype == "fp32" else 64)
    image = 730 if model == "moondream2" and dtype == "bf16" and rows <= 8 and rng.random() < 0.5 else 0
    most = 400 if dtype == "fp32" else 4000 if model == "phi2" else 9000
    high = span(16, min(2000, max(24, most // rows)) if not image else 1200)
    low = min(high, span(16, max(16, high)))
    new = span(1, {"fp32": 6}.get(dtype, 14 if model == "phi2" else 32))
    budget = rng.choice([512, 2048, 2048]) if not image else 2048
    return dict(model=model, dtype=dtype, rows=rows, image=image, low=low, high=high, new=new, budget=budget)


def prompt_ids(case):
    """Prompt ids of every request: ``low`` to ``high``, spread evenly and out of order."""
    n, low, high = case["rows"], case["low"], case["high"]
    return [low + ((i * 7 + 3) % n) * (high - low) // max(1, n - 1) for i in range(n)]


def steps_of(case):
    """The steps of a pass: ``[(request, first place, end, sampled)]`` each, prompts before decoded tokens. A request's places are
    its image, its prompt ids and the ``new - 1`` ids that follow them."""
    ends = [case["image"] + n for n in prompt_ids(case)]
    last = [e + case["new"] - 1 for e in ends]
    at = [0] * case["rows"]
    steps = []
    while any(a < b for a, b in zip(at, last)):
        left = case["budget"]
        decoded = [r for r in range(case["rows"]) if ends[r] <= at[r] < last[r]]
        left -= len(decoded)
        step = []
        for r in range(case["rows"]):
            if at[r] >= ends[r] or left <= 0:
                continue
            if at[r] == 0 and case["image"] > left:
                break                                       # (an image is one portion)
            take = min(left, ends[r] - at[r])
            if at[r] + take < ends[r]:
                aligned = (at[r] + take) // PAGE * PAGE     # (the next portion starts on a page)
                take = aligned - at[r] if aligned > max(at[r], case["image"]) else take
            step.append((r, at[r], at[r] + take, at[r] + take == ends[r]))
            left -= take
        step += [(r, at[r], at[r] + 1, True) for r in decoded]
        for r, _lo, hi, _sampled in step:
            at[r] = hi
        steps.append(step)
    return steps


# ------------------------------------------------------------------------------------------------ weights
def _route_directions(model):
    """``(directions [router outputs, width], lean [vocabulary, router outputs])``: every id leans towards as many experts as are chosen,
    in as many groups as are kept (fewer where that does not divide)."""
    s = {**_BOKORAX, **_GOZATAR}[model]
    e = s["experts"]
    outputs, (count, keep) = e["n"] + e.get("identity", 0), e["groups"]
    gen = torch.Generator("cuda").manual_seed(WEIGHTS_SEED)
    directions = torch.randn(outputs, s["width"], generator=gen, device="cuda")
    directions /= directions.norm(dim=1, keepdim=True)
    groups = next(g for g in range(keep, 0, -1) if e["top"] % g == 0)
    each = e["top"] // groups
    rand = torch.rand(VOCAB, count, outputs // count, generator=gen, device="cuda")
    group = torch.rand(VOCAB, count, generator=gen, device="cuda").topk(groups, dim=1).indices
    lean = torch.zeros(VOCAB, count, outputs // count, device="cuda")
    best = rand.topk(each, dim=2).indices
    strength = 0.20 + 0.10 * torch.rand(VOCAB, count, outputs // count, generator=gen, device="cuda")
    lean.scatter_(2, best, strength.gather(2, best))
    kept = torch.zeros(VOCAB, count, device="cuda").scatter_(1, group, 1.0)
    return directions, (lean * kept[:, :, None]).reshape(VOCAB, outputs)


def _weights(model, expected):
    """Every tensor of the model as it is stored: fp32 values of the recipe, rounded to bf16."""
    from kestrel_amd.weights import InitRecipe, random_tensor

    recipe = InitRecipe(std=0.02)
    tensors = {name: random_tensor(name, spec, WEIGHTS_SEED, recipe, device="cuda") for name, spec in expected.items()}
    if model in _BOKORAX or model in _GOZATAR:
        directions, lean = _route_directions(model)
        width = directions.shape[1]
        tensors["embed"] = tensors["embed"] * 50.0 + (lean @ directions) * width ** 0.5
        per = directions.shape[0] // {**_BOKORAX, **_GOZATAR}[model]["experts"]["groups"][0]
        for name, t in tensors.items():
            if name.endswith("mlp.router"):
                tensors[name] = torch.roll(directions, per * int(name[1:name.index(".")]), 0) * 0.35
            elif name.endswith((".norm1", ".norm2")) and model in _BOKORAX:
                tensors[name] = -0.65 + t                          # (gains are one plus what is stored)
            elif name.endswith(".w0"):
                tensors[name] = torch.linspace(-6.0, -0.5, t.numel(), device="cuda")[torch.arange(t.numel(), device="cuda") * 997 % t.numel()]
    return {name: t.to(torch.bfloat16) for name, t in tensors.items()}


_ENGINE = {}          # the one engine that is loaded, as a program keeps it; another case's replaces it


def _engine(case):
    from kestrel_amd.config import get_spec
    from kestrel_amd.engine.loading import make_runner
    from kestrel_amd.models import DecoderModel

    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _ENGINE:
        _ENGINE.clear()
        torch.cuda.empty_cache()
        device = torch.device("cuda:0")
        dtype = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
        registered, config = CONFIGS[case["model"]]
        spec = get_spec(registered)
        net = DecoderModel(spec.build_plan(spec.read_config(config)))
        net.bind({name: t.to(dtype) for name, t in _weights(case["model"], net.params()).items()}, dtype, device)
        longest = case["image"] + case["high"] + case["new"]
        runner = make_runner(net, PAGE, case["rows"] * -(-longest // PAGE), case["rows"], max_tokens_per_step=case["budget"],
                             enable_graphs=True, max_positions=longest)
        runner.prepare(case["budget"], wanted_rows=case["rows"])
        _ENGINE[key] = runner
    return _ENGINE[key]


# ------------------------------------------------------------------------------------------------ a pass
def _inputs(case, seed):
    """Ids of every request (its prompt's and those that follow) and its image."""
    rng = np.random.RandomState(seed % (1 << 32))
    ids = [rng.randint(0, VOCAB, n + case["new"] - 1) for n in prompt_ids(case)]
    gen = torch.Generator("cuda").manual_seed(seed)
    dim = CONFIGS[case["model"]][1]["text"]["dim"] if case["image"] else 0
    images = [torch.randn(case["image"], dim, generator=gen, device="cuda") for _ in ids] if case["image"] else None
    return ids, images


def prepare(case, seed):
    runner = _engine(case)
    ids, images = _inputs(case, seed)
    places = sum(sampled for step in steps_of(case) for _r, _lo, _hi, sampled in step)
    logits = torch.empty(places, VOCAB, dtype=torch.float32, device="cuda")
    return {"case": case, "runner": runner, "ids": [i.tolist() for i in ids], "images": images, "steps": steps_of(case), "logits": logits}


def run(state):
    from kestrel_amd import StepEntry

    case, runner, ids, images = state["case"], state["runner"], state["ids"], state["images"]
    image, budget, out = case["image"], case["budget"], state["logits"]
    last = [image + len(i) for i in ids]
    slots, done = {}, 0
    for step in state["steps"]:
        entries = []
        for r, lo, hi, sampled in step:
            if lo == 0:
                slots[r] = runner.admit(last[r], budget)
            tokens, embeds, blocks = ids[r][max(0, lo - image):hi - image], None, ()
            if lo < image:
                tokens, embeds, blocks = [-1] * image + tokens, images[r], ((0, image),)
            entries.append(StepEntry(slots[r], tokens, want=(hi - lo - 1,) if sampled else (), embeds=embeds, bidirectional=blocks))
        logits = runner.step(entries)
        out[done:done + logits.shape[0]].copy_(logits)       # (the next step overwrites them)
        done += logits.shape[0]
        for r, _lo, hi, _sampled in step:
            if hi == last[r]:
                runner.release(slots.pop(r))
    return out


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _facts(model):
    """``(weights every token multiplies with, [(experts, chosen, weights of one)], attention [(multiply-adds per query and key, numbers
    cached per key, window)], numbers of recurrent state, multiply-adds of the recurrences per token, width)`` without the head."""
    if model in ("moondream2", "phi2"):
        c = CONFIGS[model][1]["text"]
        d, n = c["dim"], c["n_layers"]
        return n * (4 * d * d + 2 * d * c["ff_dim"]), [], [(2 * d, 2 * d, None)] * n, 0, 0, d
    s = {**_BOKORAX, **_GOZATAR}[model]
    w, h, g, d, e = s["width"], s["heads"], s["kv_heads"], s["head"], s["experts"]
    dense, experts, attention, state, steps = 0, [], [], 0, 0
    for kind in s["order"]:
        if model in _GOZATAR:
            rh, rd, rdv = s["recurrence"]
            dense += w * (h + 2 * g) * d + h * d * w + w * (2 * rh * rd + 2 * rh * rdv + s["rank"]) + s["rank"] * rh * rd + rh * rdv * w
            attention.append((2 * h * d, 2 * g * d, s["window"]))
            state += rh * rd * rdv
            steps += 2 * rh * rd * rdv
            if kind == "d":
                dense += 2 * w * s["dense"]
                continue
        elif kind == "w":
            mh, md = s["memory"]
            dense += 5 * w * mh * md + s["rank"] * (w + mh * md)
            state += mh * md * md
            steps += 2 * mh * md * md
        else:
            keys = {"1": 1, "2": 2, "s": 0}[kind]
            dense += 2 * w * h * d + keys * w * g * d
            attention.append((2 * h * d, 0 if kind == "s" else 2 * g * d, s["window"] if kind == "1" else None))
        dense += w * (e["n"] + e.get("identity", 0)) + 3 * w * e["shared"]
        experts.append((e["n"] + e.get("identity", 0), e["top"], 3 * w * e["ff"]))
    return dense, experts, attention, state, steps, w


def work(case):
    """Bytes: every step reads each weight that its tokens use once (steps follow one another, and no cache holds a
    model), the cached keys and values its tokens see, recurrent state, and writes the logits. Operations: two per multiply-add
    of the linears, of score and value products over the keys each place sees, and of the recurrences."""
    dense, experts, attention, state, memory, width = _facts(case["model"])
    size = 4 if case["dtype"] == "fp32" else 2
    moved = flops = 0.0
    for step in steps_of(case):
        tokens = sum(hi - lo for _r, lo, hi, _s in step)
        sampled = sum(s for _r, _lo, _hi, s in step)
        used = sum(weights * n * (1.0 - (1.0 - top / n) ** tokens) for n, top, weights in experts)
        moved += size * (dense + used + (width * VOCAB if sampled else 0)) + 4.0 * sampled * VOCAB + 4.0 * width * tokens
        moved += 2 * 4.0 * state * len(step)
        flops += 2.0 * tokens * (dense + memory + sum(top * weights for _n, top, weights in experts)) + 2.0 * sampled * width * VOCAB
        for _r, lo, hi, _s in step:
            for per_pair, held, window in attention:
                window = window or hi
                moved += size * held * (hi - max(0, lo + 1 - window))
                pairs = sum(min(p + 1, window) for p in range(lo, hi))
                if lo < case["image"]:
                    pairs += case["image"] * (case["image"] - 1) // 2        # (an image's places see each other both ways)
                flops += 2.0 * per_pair * pairs
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """About four times what the path is off from 64 bits: 1.4e-6 in fp32; in bf16 0.0045 for Moondream, 0.003 for Bokorax (0.011 for a few
    tokens), 0.012 for Gozatar, whose streams carry several sublayers' roundings each."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": 0.018 if case["model"] in ("moondream2", "phi2") else 0.03}


# ------------------------------------------------------------------------------------------------ in 64 bits
def _rms(y, eps):
    return y / torch.sqrt((y * y).mean(dim=-1, keepdim=True) + eps)


def _layer_norm(x, weight, bias, eps):
    centred = x - x.mean(dim=-1, keepdim=True)
    y = centred / torch.sqrt((centred * centred).mean(dim=-1, keepdim=True) + eps) * weight
    return y if bias is None else y + bias


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _rotate(x, dims, base, factor=1.0):
    """``x`` ``[n, heads, d]``: channels ``i`` and ``i + dims / 2`` turn by ``place * base^(-2i / dims) / factor``."""
    half = dims // 2
    freqs = base ** (-2.0 * torch.arange(half, dtype=F64, device=x.device) / dims) / factor
    angle = torch.arange(x.shape[0], dtype=F64, device=x.device)[:, None, None] * freqs
    c, s = torch.cos(angle), torch.sin(angle)
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], dim=-1)


def _attend(q, k, v, scale, window=None, block=0, cap=None, sinks=None):
    """``q`` ``[n, H, d]``, ``k`` and ``v`` ``[n, G, d]``: causal (a window; the first ``block`` places see each other), ``[n, H d]``."""
    n, heads, _d = q.shape
    i, j = torch.arange(n, device=q.device)[:, None], torch.arange(n, device=q.device)[None, :]
    seen = (j <= i) & (i - j < (window or n)) | (i < block) & (j < block)
    out = torch.empty(n, heads, v.shape[2], dtype=F64, device=q.device)
    for h in range(heads):
        g = h // (heads // k.shape[1])
        s = (q[:, h] @ k[:, g].T) * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(~seen, -math.inf)
        top = s.max(dim=-1, keepdim=True).values
        if sinks is not None:
            top = torch.clamp(top, min=float(sinks[h]))
        e = torch.exp(s - top)
        total = e.sum(dim=-1, keepdim=True)
        if sinks is not None:
            total = total + torch.exp(sinks[h] - top)
        out[:, h] = (e / total) @ v[:, g]
    return out.reshape(n, -1)


def _expert(h, w, p, limit=None):
    g, u = h @ w(p + "gate").T, h @ w(p + "up").T
    if limit is None:
        return (_silu(g) * u) @ w(p + "down").T
    g, u = torch.clamp(g, max=limit), torch.clamp(u, -limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(p + "down").T


def _experts(h, w, p, m, sigmoid):
    r = m["router"]
    z = h @ w(p + "router").T
    s = torch.sigmoid(z) if sigmoid else torch.softmax(z, dim=-1)
    choice = s + w(p + "correction")
    count, keep = r["groups"]["count"], r["groups"]["keep"]
    per = choice.shape[1] // count
    best = choice.reshape(-1, count, per).topk(2 if sigmoid else 1, dim=-1).values.sum(dim=-1)
    allowed = torch.zeros_like(best, dtype=torch.bool).scatter_(1, best.topk(keep, dim=-1).indices, True)
    chosen = choice.masked_fill(~allowed.repeat_interleave(per, dim=1), -math.inf).topk(r["top"], dim=-1).indices
    picked = s.gather(1, chosen)
    weights = picked / (picked.sum(dim=-1, keepdim=True) + 1e-20) * r.get("scale", 1.0)
    out = torch.zeros_like(h)
    for e in range(choice.shape[1]):
        rows = (chosen == e).any(dim=-1).nonzero()[:, 0]
        if rows.numel():
            y = _expert(h[rows], w, f"{p}e{e}.", m["expert"].get("limit")) if e < r["experts"] else h[rows]
            out[rows] += (weights * (chosen == e)).sum(dim=-1)[rows, None] * y
    shared = _expert(h, w, p + "shared.", m["shared"].get("limit"))
    return out + (shared if sigmoid else torch.sigmoid(h @ w(p + "shared.sg").T) * shared)


def _moondream(c, w, pieces, prefix):
    """``pieces``: the embedded places of every request. Returns the normed stream of every request."""
    d, heads, eps = c["dim"], c["n_heads"], c["layer_norm_eps"]
    hd, cuts = d // heads, [p.shape[0] for p in pieces]
    rot = c.get("rotary_dim", hd // 2)
    x = torch.cat(pieces)
    for i in range(c["n_layers"]):
        p = f"text.blocks.{i}."
        h = _layer_norm(x, w(p + "ln.weight"), w(p + "ln.bias"), eps)
        parts = []
        for one in (h @ w(p + "attn.qkv.weight").T + w(p + "attn.qkv.bias")).split(cuts):
            q, k, v = one.reshape(-1, 3, heads, hd).unbind(1)
            parts.append(_attend(_rotate(q, rot, c["rope_theta"]), _rotate(k, rot, c["rope_theta"]), v, hd ** -0.5, block=prefix))
        x = x + torch.cat(parts) @ w(p + "attn.proj.weight").T + w(p + "attn.proj.bias") \
            + _gelu(h @ w(p + "mlp.fc1.weight").T + w(p + "mlp.fc1.bias")) @ w(p + "mlp.fc2.weight").T + w(p + "mlp.fc2.bias")
    return _layer_norm(x, w("text.post_ln.weight"), w("text.post_ln.bias"), eps).split(cuts)


def _decaying_memory(x, w, p, m, eps):
    n, (heads, d) = x.shape[0], (m["heads"], m["dim"])
    before = torch.cat([torch.zeros_like(x[:1]), x[:-1]])
    mixes = {s: x + (before - x) * w(p + "mu." + s) for s in "rkvgw"}
    r, k, v = ((mixes[s] @ w(p + s).T).reshape(n, heads, d) for s in "rkv")
    decay = torch.exp(-torch.exp(torch.tanh(mixes["w"] @ w(p + "w1").T) @ w(p + "w2").T + w(p + "w0"))).reshape(n, heads, d)
    bonus = ((r * w(p + "u").reshape(heads, d) * k).sum(dim=-1, keepdim=True)) * v
    state, out = torch.zeros(heads, d, d, dtype=F64, device=x.device), torch.empty_like(v)
    for t in range(n):
        torch.sum(state * r[t][:, :, None], dim=1, out=out[t])
        state.mul_(decay[t][:, :, None]).addcmul_(k[t][:, :, None], v[t][:, None, :])
    o = _rms(out + bonus, eps).reshape(n, -1) * w(p + "norm") * _silu(mixes["g"] @ w(p + "g").T)
    return o @ w(p + "o").T


def _bokorax(c, w, pieces):
    eps, cuts, kept = c["norm"]["eps"], [p.shape[0] for p in pieces], {}
    x = torch.cat(pieces) * c["embedding"]["scale"]
    for i, layer in enumerate(c["layers"]):
        p, m, parts = f"l{i}.mix.", layer["mixer"], []
        if layer["type"] != "wkv":
            heads, kv, d, rot = m["heads"], m["kv_heads"], m["dim"], m["rot"]
            turn = (rot["dims"], rot["base"], rot.get("scaling", {}).get("factor", 1.0))
        for r, one in enumerate(x.split(cuts)):
            if layer["type"] == "wkv":
                parts.append(_decaying_memory(one, w, p, m, eps))
                continue
            q = one @ w(p + "q").T
            if layer["type"] == "attention":
                k = one @ w(p + "k").T
                v = k.reshape(-1, kv, d)
                q, k = _rms(q, eps) * w(p + "q.norm"), _rms(k, eps) * w(p + "k.norm")
                o = _attend(_rotate(q.reshape(-1, heads, d), *turn), _rotate(k.reshape(-1, kv, d), *turn), v, m["scale"], window=m["mask"]["size"])
            else:
                q = _rotate(_rms(q.reshape(-1, heads, d), eps) * w(p + "q.norm"), *turn)
                if "kv_from" not in m:
                    k = _rotate(_rms((one @ w(p + "k").T).reshape(-1, kv, d), eps) * w(p + "k.norm"), *turn)
                    kept[i, r] = k, (one @ w(p + "v").T).reshape(-1, kv, d)
                o = _attend(q, *kept[m.get("kv_from", i), r], m["scale"], cap=m["softcap"], sinks=w(p + "sink"))
                o = (o.reshape(-1, heads, d) * torch.sigmoid(one @ w(p + "g").T)[:, :, None]).reshape(-1, heads * d)
            parts.append(o @ w(p + "o").T)
        x = x + _rms(torch.cat(parts), eps) * (1.0 + w(f"l{i}.norm1"))
        x = x + _rms(_experts(x, w, f"l{i}.mlp.", layer["mlp"], False), eps) * (1.0 + w(f"l{i}.norm2"))
    return (_rms(x, eps) * (1.0 + w("final.norm"))).split(cuts)


def _convolved(y, taps):
    n, k = y.shape[0], taps.shape[1]
    padded = torch.cat([torch.zeros(k - 1, y.shape[1], dtype=F64, device=y.device), y])
    return sum(padded[j:j + n] * taps[:, j] for j in range(k))


def _gozatar_mixer(h, w, p, m, eps):
    n, a, r = h.shape[0], m["left"], m["right"]
    q, k, v = (_convolved(h @ w(p + "left." + s).T, w(p + "left." + s + ".conv")) for s in "qkv")
    q, k = (_rms(_rotate(y.reshape(n, -1, a["dim"]), a["rot"]["dims"], a["rot"]["base"]), eps) for y in (q, k))
    left = _attend(q, k, v.reshape(n, -1, a["vdim"]), a["scale"], window=a["mask"]["size"]) @ w(p + "left.o").T
    p += "right."
    heads, d, dv = r["heads"], r["dim"], r["vdim"]
    q, k = (h @ w(p + "q").T).reshape(n, heads, d) * d ** -0.5, (h @ w(p + "k").T).reshape(n, heads, d)
    v = (h @ w(p + "v").T).reshape(n, heads, dv)
    decay = (torch.sigmoid((h @ w(p + "a1").T) @ w(p + "a2").T + w(p + "a2.b")) ** (1.0 / r["tau"])).reshape(n, heads, d)
    state, out = torch.zeros(heads, d, dv, dtype=F64, device=h.device), torch.empty_like(v)
    for t in range(n):
        state.mul_(decay[t][:, :, None]).addcmul_(k[t][:, :, None], v[t][:, None, :])
        torch.sum(state * q[t][:, :, None], dim=1, out=out[t])
    o = (_rms(out, eps) * w(p + "norm")).reshape(n, -1) * _silu(h @ w(p + "g").T)
    return m["left_scale"] * left + m["right_scale"] * (o @ w(p + "o").T)


def _gozatar(c, w, pieces):
    eps, cuts, count = c["norm"]["eps"], [p.shape[0] for p in pieces], c["streams"]
    streams = torch.cat(pieces).expand(count, -1, -1)
    for i, layer in enumerate(c["layers"]):
        for half in ("1", "2"):
            h = _layer_norm((w(f"l{i}.hc{half}.in")[:, None, None] * streams).sum(dim=0), w(f"l{i}.norm{half}"), None, eps)
            if half == "1":
                y = torch.cat([_gozatar_mixer(one, w, f"l{i}.mix.", layer["mixer"], eps) for one in h.split(cuts)])
            elif layer["mlp"]["kind"] == "dense":
                y = _gelu(h @ w(f"l{i}.mlp.up").T) @ w(f"l{i}.mlp.down").T
            else:
                y = _experts(h, w, f"l{i}.mlp.", layer["mlp"], True)
            mix, out = w(f"l{i}.hc{half}.mix"), w(f"l{i}.hc{half}.out")
            streams = torch.einsum("st,snw->tnw", mix, streams) + out[:, None, None] * y
    return _layer_norm(streams.sum(dim=0), w("final.norm"), None, eps).split(cuts)


@torch.no_grad()
def exact(case, seed):
    """The logits of the sampled places from whole sequences without a cache, in 64 bits from the stored weights."""
    from kestrel_amd.config import get_spec
    from kestrel_amd.models import DecoderModel

    _ENGINE.clear()
    torch.cuda.empty_cache()
    registered, config = CONFIGS[case["model"]]
    spec = get_spec(registered)
    stored = _weights(case["model"], DecoderModel(spec.build_plan(spec.read_config(config))).params())   # (their names and shapes)
    w = lambda name: stored[name].to(F64)  # noqa: E731
    ids, images = _inputs(case, seed)
    table = stored["text.wte" if registered == "moondream2" else "embed"]
    pieces = [table[torch.from_numpy(i).cuda()].to(F64) for i in ids]
    if images is not None:
        pieces = [torch.cat([image.to(F64), piece]) for image, piece in zip(images, pieces)]
    if registered == "moondream2":
        normed = _moondream(config["text"], w, pieces, case["image"])
    else:
        normed = (_bokorax if registered == "bokorax" else _gozatar)(config, w, pieces)
    rows = torch.stack([normed[r][hi - 1] for step in steps_of(case) for r, _lo, hi, sampled in step if sampled])
    if registered == "moondream2":
        return rows @ w("text.lm_head.weight").T + w("text.lm_head.bias")
    return rows @ w("head").T
