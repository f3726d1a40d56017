"""A block: a mixer, a feed-forward and their norm(s) in one of the known arrangements."""

from __future__ import annotations

from typing import Callable, Dict, Optional

import torch

from .base import LayerCache, Part, SideLinear, build_part
from .specs import LayerSpec, ParamSpec
from .streams import StreamReading


def _parallel_few_rows(block: "Block", x, batch, cache, normed, then, handed) -> bool:
    """The parallel block for a few bf16 rows in three launches: norm + both first linears, the
    mixer's core, both last linears + residual. Needs a mixer and a feed-forward that offer their
    stages (``input_projection`` / ``output_projection``); returns ``False`` otherwise. More rows, as long as either the two first linears are
    faster in one launch (``fast.joint_tile``) or the two last ones and the norm behind them as one product of tiles (``fast.pair_tiles_pay``,
    ``fast.pair_large_parts``): what is not is launches of its own then, and a gated feed-forward keeps to its ``forward``, which has a better way for many rows.
    ``normed``: the block's norm of ``x``, where the block before has computed it; ``then``: the norm
    the next block starts with, which the last launch computes as well where it pays (``handed``, a
    list, then gets the normalised rows)."""
    from ..ops import fast
    from ..ops.linear import ACT_GATED, linear

    n = x.shape[0]
    if block.dtype != torch.bfloat16 or block.feed_forward is None:
        return False
    m_in, f_in = block.mixer.input_projection(), block.feed_forward.input_projection()
    m_out, f_out = block.mixer.output_projection(), block.feed_forward.output_projection()
    if m_in is None or f_in is None or m_out is None or f_out is None:
        return False
    sizes = (n, x.shape[1], m_out[0].shape[1], f_out[0].shape[1])
    many = n > fast.SKINNY_MAX_ROWS
    # (the large tiles only in front of a norm that their finishing launch takes along)
    large = many and then is not None and then.layernorm_operands() is not None and fast.pair_large_parts(*sizes) > 0
    if many and (f_in[3] & ACT_GATED or not (large or fast.pair_tiles_pay(*sizes, True) or
                                             fast.joint_tile(n, m_in[0].shape[0], f_in[0].shape[0], x.shape[1]))):
        return False
    ws = batch.workspace
    projected = ws.get("block.mixer_in", (n, m_in[2]), block.dtype)
    hidden = ws.get("block.ff_hidden", (n, f_in[2]), block.dtype)
    norm = block.norm
    fused = False
    beside = None
    if normed is not None:
        fused = fast.linear_two_outputs(normed, m_in[0], m_in[1], projected, 0, f_in[0], f_in[1], hidden, f_in[3])
    ln = norm.layernorm_operands()            # (a norm of another form is run through its own forward below)
    rms = norm.rms_operands() if ln is None and callable(getattr(norm, "rms_operands", None)) else None
    if not fused and fast.FUSE_LAYERNORM_PROLOGUE and rms is not None:
        # a root-mean-square norm in the prologue of the launch that projects for the mixer and the feed-forward
        fused = fast.layernorm_linear(x, rms[0], None, rms[1], m_in[0], m_in[1], projected, 0, f_in[0], f_in[1], hidden, f_in[3],
                                      centred=False)
    if not fused and fast.FUSE_LAYERNORM_PROLOGUE and ln is not None:
        # the feed-forward's first linear goes into the mixer's launch where the mixer takes it (the
        # launch of the mixer's first linear then leaves the normalised rows for it), else into the
        # launch of the mixer's first linear
        h = ws.get("block.h", tuple(x.shape), block.dtype)
        job = SideLinear(h, f_in[0], f_in[1], hidden, f_in[3])
        if block.mixer.takes_beside(job, batch, cache) and \
                fast.layernorm_linear(x, *ln, m_in[0], m_in[1], projected, 0, store=h):
            fused, beside = True, job
        else:
            fused = fast.layernorm_linear(x, *ln, m_in[0], m_in[1], projected, 0, f_in[0], f_in[1], hidden, f_in[3])
    if not fused:
        h = normed
        if h is None:
            h = ws.get("block.h", tuple(x.shape), block.dtype)
            norm.forward(x, h)
        first = (h, m_in[0], m_in[1], projected, 0, f_in[0], f_in[1], hidden, f_in[3])
        if not (fast.linear_joint(*first) if many else fast.linear_two_outputs(*first)):
            linear(h, m_in[0], m_in[1], projected)
            linear(h, f_in[0], f_in[1], hidden, act=f_in[3])
    mixed = block.mixer.attend(projected, batch, cache, beside) if beside is not None \
        else block.mixer.attend(projected, batch, cache)
    # More rows than the next block's first launch normalises by itself, or a last launch of this block that
    # ends in a kernel that finishes whole rows anyway: the next block's norm is computed here, by that
    # kernel, instead of in a launch or a prologue of its own (9 to 16 rows of 2048: 1 to 2 % of a step;
    # rows of 2560, which leave the prologue's kernel no registers for a third strip of weights in flight, from
    # 5 rows on: 3 to 4 %).
    handing = n > fast.SKINNY_LN_MAX_ROWS or fast.pair_finishes_rows(n, x.shape[1])
    then_ln = then.layernorm_operands() if then is not None and handing and (not many or large or fast.pair_tiles_pay(*sizes, True)) else None
    if then_ln is not None:
        rows = ws.get("block.handed", tuple(x.shape), block.dtype)
        if fast.linear_pair_accumulate(mixed, m_out[0], m_out[1], hidden, f_out[0], f_out[1], x,
                                       then_norm=(*then_ln, rows), large=large):
            handed.append(rows)
            return True
    pays = not many or fast.pair_tiles_pay(*sizes, False)
    if not (pays and fast.linear_pair_accumulate(mixed, m_out[0], m_out[1], hidden, f_out[0], f_out[1], x)):
        linear(mixed, m_out[0], m_out[1], x, accumulate=True)
        linear(hidden, f_out[0], f_out[1], x, accumulate=True)
    return True


def _parallel_few_rows_f32(block: "Block", x, batch, cache, normed) -> bool:
    """The parallel block for a few fp32 rows in three launches, as ``_parallel_few_rows`` has them: norm and both first linears, the mixer's core, both last
    linears; what ``ops.core`` does not cover is a launch each. Returns ``False`` (nothing was run) where the parts do not offer their stages."""
    from ..ops import core
    from ..ops.linear import ACT_GATED, linear

    n = x.shape[0]
    if block.dtype != torch.float32 or n > core.FEW_F32_ROWS or block.feed_forward is None:
        return False
    m_in, f_in = block.mixer.input_projection(), block.feed_forward.input_projection()
    m_out, f_out = block.mixer.output_projection(), block.feed_forward.output_projection()
    if m_in is None or f_in is None or m_out is None or f_out is None or f_in[3] & ACT_GATED:
        return False
    ws = batch.workspace
    projected = ws.get("block.mixer_in", (n, m_in[2]), block.dtype)
    hidden = ws.get("block.ff_hidden", (n, f_in[2]), block.dtype)
    first = (m_in[0], m_in[1], projected, 0, f_in[0], f_in[1], hidden, f_in[3])
    ln = block.norm.layernorm_operands() if normed is None else None
    if ln is None or not core.linears_first_f32(x, ln, *first):
        h = normed
        if h is None:
            h = ws.get("block.h", tuple(x.shape), block.dtype)
            block.norm.forward(x, h)
        if not core.linears_first_f32(h, None, *first):
            linear(h, m_in[0], m_in[1], projected)
            linear(h, f_in[0], f_in[1], hidden, act=f_in[3])
    mixed = block.mixer.attend(projected, batch, cache)
    if not core.linears_last_f32(mixed, m_out[0], m_out[1], hidden, f_out[0], f_out[1], x):
        linear(mixed, m_out[0], m_out[1], x, accumulate=True)
        linear(hidden, f_out[0], f_out[1], x, accumulate=True)
    return True


def _parallel_wanted(block: "Block", x, batch, cache, normed, wanted):
    """The parallel block that leaves the wanted tokens alone: the mixer's first linear and what it keeps of all tokens, everything else for those."""
    from ..ops import fast
    from ..ops.linear import linear

    ff, ws = block.feed_forward, batch.workspace
    h = normed
    if h is None:
        h = ws.get("block.h", tuple(x.shape), block.dtype)
        block.norm.forward(x, h)
    few, h_few = wanted.buffer("x", x), wanted.buffer("h", h)
    m_out = block.mixer.output_projection() if callable(getattr(block.mixer, "attend_wanted", None)) else None
    f_in, f_out = (ff.input_projection(), ff.output_projection()) if ff is not None else (None, None)
    if m_out is None:
        # (a mixer that only adds: into the stream of all tokens)
        wanted.gather((h, h_few))
        block.mixer.forward(h, batch, cache, x)
        wanted.gather((x, few))
        mixed = None
    else:
        mixed = block.mixer.attend_wanted(block.mixer.project(h, batch), batch, cache, wanted, (x, few), (h, h_few))
    if wanted.count == 0:
        return few, None
    if mixed is not None and f_in is not None and f_out is not None:
        hidden = ws.get("block.ff_hidden", (wanted.count, f_in[2]), block.dtype)
        linear(h_few, f_in[0], f_in[1], hidden, act=f_in[3])
        if block.dtype == torch.bfloat16 and fast.linear_pair_accumulate(mixed, m_out[0], m_out[1], hidden, f_out[0], f_out[1], few):
            return few, None
        linear(mixed, m_out[0], m_out[1], few, accumulate=True)
        linear(hidden, f_out[0], f_out[1], few, accumulate=True)
        return few, None
    if mixed is not None:
        linear(mixed, m_out[0], m_out[1], few, accumulate=True)
    if ff is not None:
        ff.forward(h_few, wanted.batch, few)
    return few, None


def _parallel(block: "Block", x, batch, cache, normed=None, then=None, wanted=None):
    """``x + mixer(norm(x)) + ff(norm(x))``: both branches read the same normalised input (a block without a
    feed-forward has the first branch only).

    Reference: ``kestrel/models/moondream/text.py:222-275``.
    """
    if wanted is not None:
        return _parallel_wanted(block, x, batch, cache, normed, wanted)
    handed = []
    if _parallel_few_rows(block, x, batch, cache, normed, then, handed):
        return handed[0] if handed else None
    if _parallel_few_rows_f32(block, x, batch, cache, normed):
        return None
    h = normed
    if h is None:
        h = batch.workspace.get("block.h", tuple(x.shape), block.dtype)
        block.norm.forward(x, h)
    block.mixer.forward(h, batch, cache, x)
    if block.feed_forward is not None:
        block.feed_forward.forward(h, batch, x)
    return None


_parallel.hands_over = _parallel.narrows = True


def _sequential_few_rows(block: "Block", x, batch, cache) -> bool:
    """The sequential block for a few bf16 rows: each norm in the prologue of the launch that reads it (the mixer's first
    linear; the feed-forward's first linear where it offers ``from_stream``). Needs a root-mean-square norm and a mixer
    that offers its stages; returns ``False`` (nothing was run) otherwise."""
    from ..ops import fast
    from ..ops.linear import linear

    n = x.shape[0]
    if block.dtype != torch.bfloat16 or n > fast.SKINNY_LN_MAX_ROWS or not fast.FUSE_LAYERNORM_PROLOGUE:
        return False
    rms = block.norm.rms_operands() if callable(getattr(block.norm, "rms_operands", None)) else None
    m_in, m_out = block.mixer.input_projection(), block.mixer.output_projection()
    if rms is None or m_in is None or m_out is None:
        return False
    ws = batch.workspace
    projected = ws.get("block.mixer_in", (n, m_in[2]), block.dtype)
    if not fast.layernorm_linear(x, rms[0], None, rms[1], m_in[0], m_in[1], projected, 0, centred=False):
        return False
    linear(block.mixer.attend(projected, batch, cache), m_out[0], m_out[1], x, accumulate=True)
    if block.feed_forward is not None:
        from_stream = getattr(block.feed_forward, "from_stream", None)
        if from_stream is None or not from_stream(x, block.norm2, batch):
            h = ws.get("block.h", tuple(x.shape), block.dtype)
            block.norm2.forward(x, h)
            block.feed_forward.forward(h, batch, x)
    return True


def _sequential(block: "Block", x, batch, cache) -> None:
    """``x += mixer(norm(x)); x += ff(norm2(x))``; without a feed-forward the first half only."""
    if _sequential_few_rows(block, x, batch, cache):
        return
    h = batch.workspace.get("block.h", tuple(x.shape), block.dtype)
    block.norm.forward(x, h)
    block.mixer.forward(h, batch, cache, x)
    if block.feed_forward is not None:
        block.norm2.forward(x, h)
        block.feed_forward.forward(h, batch, x)


# Whether a block of weighted branches leaves the sum ``x += scale * delta`` to whoever reads the stream next (the
# next such block adds it in the pass that computes its norms; anything else calls ``settle`` first) instead of
# adding it in a launch of its own. Off: every block leaves the stream complete (what a test that reads the
# stream between blocks needs).
DEFER_RESIDUAL = True
_PENDING = "residual_pending"


def settle(x, batch) -> None:
    """Add what a block before has left to be added into the fp32 stream ``x``."""
    from ..ops import core

    host = getattr(batch, "host", None)
    pending = host.pop(_PENDING, None) if host else None
    if pending is not None:
        core.add_scaled(x, pending[0], pending[1])


def _two_branches_by_stages(block: "Block", h1, h2, batch, cache, delta) -> bool:
    """Both branches through the stages that mixer and feed-forward offer, so that the first of the last linears
    writes ``delta`` and nobody has to clear it: for a few bf16 rows, and where it pays for more (``fast.pair_tiles_pay``), the
    two last linears are one product.
    ``False``: a part offers no stages (its ``forward`` then adds into a cleared ``delta``)."""
    from ..ops import fast
    from ..ops.linear import linear

    n = h1.shape[0]
    ff = block.feed_forward
    m_in, m_out = block.mixer.input_projection(), block.mixer.output_projection()
    f_in, f_out = (ff.input_projection(), ff.output_projection()) if ff is not None else (None, None)
    if m_in is None or m_out is None or (ff is not None and (f_in is None or f_out is None)):
        return False
    ws = batch.workspace
    projected = ws.get("block.mixer_in", (n, m_in[2]), block.dtype)
    linear(h1, m_in[0], m_in[1], projected)
    hidden = None
    if ff is not None:
        hidden = ws.get("block.ff_hidden", (n, f_in[2]), block.dtype)
        linear(h2, f_in[0], f_in[1], hidden, act=f_in[3])
    mixed = block.mixer.attend(projected, batch, cache)
    if ff is not None and block.dtype == torch.bfloat16 and \
            (n <= fast.SKINNY_MAX_ROWS or fast.pair_tiles_pay(n, delta.shape[1], m_out[0].shape[1], f_out[0].shape[1], False)) and \
            fast.linear_pair_accumulate(mixed, m_out[0], m_out[1], hidden, f_out[0], f_out[1], delta, accumulate=False):
        return True
    linear(mixed, m_out[0], m_out[1], delta)
    if ff is not None:
        linear(hidden, f_out[0], f_out[1], delta, accumulate=True)
    return True


def _parallel_two_norms(block: "Block", x, batch, cache) -> None:
    """``x + residual_scale * (mixer(norm(x)) + ff(norm2(x)))``: two branches, each with a norm of its own of the
    same ``x``; without a feed-forward, ``x + residual_scale * mixer(norm(x))``.

    Both norms come from one pass over ``x`` where they are LayerNorms of one eps; that pass also adds what the
    block before has left to be added (``DEFER_RESIDUAL``). The branches' sum is kept in a buffer of its own and
    enters the stream with the weight in fp32, like the stream."""
    from ..ops import core

    ws = batch.workspace
    h1 = ws.get("block.h", tuple(x.shape), block.dtype)
    delta = ws.get("block.delta", tuple(x.shape), torch.float32)
    ff = block.feed_forward
    ln1 = block.norm.layernorm_operands()
    ln2 = block.norm2.layernorm_operands() if ff is not None else None
    h2 = ws.get("block.h2", tuple(x.shape), block.dtype) if ff is not None else None
    host = batch.host
    pending = host.get(_PENDING)
    if pending is not None and pending[0].data_ptr() != delta.data_ptr():
        settle(x, batch)              # (left in another buffer than this block's)
        pending = None
    # parts that offer their stages write the buffer; parts that only add need it cleared
    staged = block.mixer.input_projection() is not None and block.mixer.output_projection() is not None and \
        (ff is None or (ff.input_projection() is not None and ff.output_projection() is not None))
    sum_args = dict(delta=delta if (pending is not None or not staged) else None, scale=pending[1] if pending else 1.0,
                    apply=pending is not None, clear=not staged)
    if ln1 is not None and (ff is None or (ln2 is not None and float(ln2[2]) == float(ln1[2]))):
        core.layernorm_pair(x, ln1, ln2, h1, h2, **sum_args)
    else:
        core.layernorm_pair(x, None, None, None, None, **sum_args)
        block.norm.forward(x, h1)
        if ff is not None:
            block.norm2.forward(x, h2)
    host.pop(_PENDING, None)
    if not (staged and _two_branches_by_stages(block, h1, h2, batch, cache, delta)):
        block.mixer.forward(h1, batch, cache, delta)
        if ff is not None:
            ff.forward(h2, batch, delta)
    if DEFER_RESIDUAL:
        host[_PENDING] = (delta, float(block.spec.residual_scale))
    else:
        core.add_scaled(x, delta, block.spec.residual_scale)


_parallel_two_norms.defers = True


class StreamRounding:
    """What a block of the arrangement ``output_norms`` reads first: the stream itself, rounded to the activation type (``wanted``) or, for a
    mixer that says ``reads_stream``, as it is. No norm: it offers no operands of one."""

    def __init__(self, wanted: bool) -> None:
        self.wanted = wanted

    def layernorm_operands(self):
        return None

    def rms_operands(self):
        return None


def _into_delta(part, delta, *operands) -> None:
    """A part's output written into fp32 ``delta``."""
    if callable(getattr(part, "mix", None)):
        part.mix(*operands, delta, False)
    else:
        delta.zero_()
        part.forward(*operands, delta)


def _mix_wanted(block: "Block", h, x, batch, cache, delta, wanted):
    """``(x, delta)`` of the wanted tokens: their rows of the stream and the mixer's output for them. The mixer leaves what later steps read of
    all tokens; one that offers ``mix_wanted`` does only that for the others."""
    few, out = wanted.buffer("x", x), wanted.buffer("delta", delta)
    if callable(getattr(block.mixer, "mix_wanted", None)):
        block.mixer.mix_wanted(h, batch, cache, out, wanted, (x, few))
    else:
        _into_delta(block.mixer, delta, h, batch, cache)
        wanted.gather((x, few), (delta, out))
    return few, out


def _output_norms(block: "Block", x, batch, cache, normed=None, then=None, wanted=None):
    """``x += norm(mixer(x)); x += norm2(ff(x))``: the parts read the stream itself (rounded to the activation type, or,
    for a mixer that says ``reads_stream``, as it is) and the norms stand behind them. Each part writes its output into
    an fp32 buffer (``mix``; a part without it adds into a cleared buffer through ``forward``); one launch normalises it, adds it
    into the stream and leaves the rounding that the next reader begins with (``normed``, from the block before). A feed-forward
    that offers ``mix_normed`` takes that launch's work into its own last one."""
    from ..ops import core

    mixer, ws = block.mixer, batch.workspace
    if wanted is not None and getattr(mixer, "only_reads", False):
        # (nobody else reads anything of a token's row here: the whole block for the wanted tokens alone)
        few = wanted.buffer("x", x)
        rows = (normed, wanted.buffer("h", normed)) if normed is not None else None
        wanted.gather((x, few), *([rows] if rows else []))
        return few, _output_norms(block, few, wanted.batch, cache, rows[1] if rows else None, then) if wanted.count else None
    delta = ws.get("block.delta", tuple(x.shape), torch.float32)
    source = x
    if block.dtype != torch.float32 and not getattr(mixer, "reads_stream", False):
        source = normed
        if source is None:
            source = ws.get("block.h", tuple(x.shape), block.dtype)
            core.cast_columns(x, source)
    if wanted is not None:
        x, delta = _mix_wanted(block, source, x, batch, cache, delta, wanted)
        return x, _output_norms_behind(block, x, wanted.batch, delta, then) if wanted.count else None
    _into_delta(mixer, delta, source, batch, cache)
    return _output_norms_behind(block, x, batch, delta, then)


def _output_norms_behind(block: "Block", x, batch, delta, then):
    """What ``_output_norms`` does behind the mixer, whose output is ``delta``."""
    from ..ops import core

    ws = batch.workspace
    rounds = block.dtype != torch.float32

    def add(norm, rows) -> bool:
        """``x += norm(delta)``, the stream's rounding into ``rows`` (``None``: not wanted); returns whether ``rows`` was written."""
        first = norm.rms_operands() if callable(getattr(norm, "rms_operands", None)) else None
        if first is not None:
            core.add_normed(x, delta, first, None, rows)
            return rows is not None
        if callable(getattr(norm, "add_normed", None)):
            norm.add_normed(delta, x)
        else:
            summed = ws.get("block.normed", tuple(x.shape), torch.float32)
            norm.forward(delta, summed)
            core.add_scaled(x, summed, 1.0)
        return False

    handed = ws.get("block.handed", tuple(x.shape), block.dtype) if rounds and isinstance(then, StreamRounding) and then.wanted else None
    ff = block.feed_forward
    if ff is None:
        return handed if add(block.norm, handed) else None
    h = x
    if rounds:
        h = ws.get("block.h2", tuple(x.shape), block.dtype)
    if not add(block.norm, h if rounds else None) and rounds:
        core.cast_columns(x, h)
    second = block.norm2.rms_operands() if callable(getattr(block.norm2, "rms_operands", None)) else None
    if callable(getattr(ff, "mix_normed", None)) and second is not None:
        ff.mix_normed(h, batch, x, second, None, handed)
        return handed
    _into_delta(ff, delta, h, batch)
    return handed if add(block.norm2, handed) else None


_output_norms.hands_over = _output_norms.narrows = True


def _add_normed(norm, delta, x, then, rows, ws) -> bool:
    """``x += norm(delta)``, and the norm ``then`` of the new rows of the stream into ``rows``, in one launch where both are
    root-mean-square norms (returns whether ``rows`` was written)."""
    from ..ops import core

    first = norm.rms_operands() if callable(getattr(norm, "rms_operands", None)) else None
    if first is None:
        if callable(getattr(norm, "add_normed", None)):
            norm.add_normed(delta, x)
        else:
            normed = ws.get("block.normed", tuple(x.shape), torch.float32)
            norm.forward(delta, normed)
            core.add_scaled(x, normed, 1.0)
        return False
    second = then.rms_operands() if then is not None and callable(getattr(then, "rms_operands", None)) else None
    core.add_normed(x, delta, first, second, rows if second is not None else None)
    return second is not None


def _norms_around(block: "Block", x, batch, cache, normed=None, then=None, wanted=None):
    """``x += norm_after(mixer(norm(x))); x += norm2_after(ff(norm2(x)))``: a norm before and behind each sublayer.

    A sublayer writes its output into an fp32 buffer (``mix``); one launch then normalises it, adds it into the stream
    and computes the norm that the next reader of the stream begins with: ``norm2`` behind the mixer, and behind the
    feed-forward the first norm of the block that follows (``then``), whose rows are handed over. A feed-forward that
    offers ``mix_normed`` takes that launch's work into its own last one."""
    delta = batch.workspace.get("block.delta", tuple(x.shape), torch.float32)
    h = normed
    if h is None:
        h = batch.workspace.get("block.h", tuple(x.shape), block.dtype)
        block.norm.forward(x, h)
    if wanted is not None:
        x, delta = _mix_wanted(block, h, x, batch, cache, delta, wanted)
        return x, _norms_around_behind(block, x, wanted.batch, delta, then) if wanted.count else None
    _into_delta(block.mixer, delta, h, batch, cache)
    return _norms_around_behind(block, x, batch, delta, then)


def _norms_around_behind(block: "Block", x, batch, delta, then):
    """What ``_norms_around`` does behind the mixer, whose output is ``delta``."""
    ws = batch.workspace
    ff = block.feed_forward
    handed = ws.get("block.handed", tuple(x.shape), block.dtype)
    if ff is None:
        return handed if _add_normed(block.norm_after, delta, x, then, handed, ws) else None
    h = ws.get("block.h2", tuple(x.shape), block.dtype)
    if not _add_normed(block.norm_after, delta, x, block.norm2, h, ws):
        block.norm2.forward(x, h)
    if callable(getattr(ff, "mix_normed", None)):
        first = block.norm2_after.rms_operands() if callable(getattr(block.norm2_after, "rms_operands", None)) else None
        second = then.rms_operands() if then is not None and callable(getattr(then, "rms_operands", None)) else None
        if first is not None:
            ff.mix_normed(h, batch, x, first, second, handed if second is not None else None)
            return handed if second is not None else None
    _into_delta(ff, delta, h, batch)
    return handed if _add_normed(block.norm2_after, delta, x, then, handed, ws) else None


_norms_around.hands_over = _norms_around.narrows = True


def _streams(block: "Block", x, batch, cache, normed=None, then=None, wanted=None):
    """The stream as several copies ``x`` ``[n, S, dim]`` (hyper-connections): ``u = sum_s in[s] x_s``, ``y = mixer(norm(u))``,
    ``x_t <- sum_s mix[s, t] x_s + out[t] y``, then the same with the feed-forward and its own numbers and norm.

    One launch stands between two sublayers: it writes the one's output into the streams and leaves the norm of what the
    next one reads (``then``, a ``StreamReading``, behind the last: its rows are handed over). A feed-forward that offers
    ``mix_streams`` takes that launch's work into its own last one, and one with ``choose_streams`` its choice into the one in front of it."""
    from ..ops import core

    n, _count, dim = x.shape
    delta = batch.workspace.get("block.delta", (n, dim), torch.float32)
    h = normed
    if h is None:
        h = batch.workspace.get("block.h", (n, dim), block.dtype)
        core.streams_step(x, reading=block.reader.operands(), h=h)
    if wanted is not None:
        x, delta = _mix_wanted(block, h, x, batch, cache, delta, wanted)
        return x, _streams_behind(block, x, wanted.batch, delta, then) if wanted.count else None
    _into_delta(block.mixer, delta, h, batch, cache)
    return _streams_behind(block, x, batch, delta, then)


def _streams_behind(block: "Block", x, batch, delta, then):
    """What ``_streams`` does behind the mixer, whose output is ``delta``."""
    from ..ops import core

    ws = batch.workspace
    n, _count, dim = x.shape
    ff = block.feed_forward
    last = then.operands() if then is not None else None
    handed = ws.get("block.handed", (n, dim), block.dtype) if then is not None else None
    if ff is None:
        core.streams_step(x, delta, block.streams.matrix, block.streams.out, last, handed)
        return handed
    h2 = ws.get("block.h2", (n, dim), block.dtype)
    reading = block.reader2.operands()
    chosen = callable(getattr(ff, "choose_streams", None)) and ff.choose_streams(x, delta, block.streams, reading, h2, batch)
    if not chosen:
        core.streams_step(x, delta, block.streams.matrix, block.streams.out, reading, h2)
    if callable(getattr(ff, "mix_streams", None)):
        ff.mix_streams(h2, batch, x, block.streams2, last, handed, **({"chosen": True} if chosen else {}))
        return handed
    _into_delta(ff, delta, h2, batch)
    core.streams_step(x, delta, block.streams2.matrix, block.streams2.out, last, handed)
    return handed


_streams.hands_over = _streams.narrows = True


ARRANGEMENTS: Dict[str, Callable] = {"parallel": _parallel, "sequential": _sequential,
                                     "parallel_two_norms": _parallel_two_norms, "output_norms": _output_norms,
                                     "norms_around": _norms_around, "streams": _streams}


def register_arrangement(name: str, fn: Callable) -> None:
    """``fn(block, x, batch, cache)`` updates the fp32 residual ``x`` in place. A function with the
    attribute ``hands_over = True`` is called as ``fn(block, x, batch, cache, normed=, then=)``:
    ``normed`` is ``block.norm`` of ``x`` if the block before has computed it (else ``None``), ``then``
    the first norm of the block that follows (or ``None``); it may return that norm of its result, or
    ``None``. One with ``narrows = True`` besides is given ``wanted=`` (a ``WantedTokens``) where only those tokens' rows are read
    behind it, and returns ``(their rows of the stream, that norm of them or None)`` then."""
    ARRANGEMENTS[name] = fn


class Block:
    """Parts of one layer, built from its specification through the registries."""

    def __init__(self, spec: LayerSpec) -> None:
        if spec.arrangement not in ARRANGEMENTS:
            raise ValueError(f"unknown arrangement {spec.arrangement!r}; known: {', '.join(sorted(ARRANGEMENTS))}")
        self.spec = spec
        self.norm = build_part("norm", spec.norm)
        self.norm2 = build_part("norm", spec.norm2) if spec.norm2 is not None else None
        if spec.arrangement == "sequential" and self.norm2 is None and spec.feed_forward is not None:
            raise ValueError("the sequential arrangement needs norm2 for its feed-forward")
        self.norm_after = build_part("norm", spec.norm_after) if getattr(spec, "norm_after", None) is not None else None
        self.norm2_after = build_part("norm", spec.norm2_after) if getattr(spec, "norm2_after", None) is not None else None
        if spec.arrangement == "norms_around" and (self.norm_after is None or (
                spec.feed_forward is not None and (self.norm2 is None or self.norm2_after is None))):
            raise ValueError("the norms_around arrangement needs norm_after, and norm2 and norm2_after for its feed-forward")
        self.streams = build_part("stream_mix", spec.streams) if getattr(spec, "streams", None) is not None else None
        self.streams2 = build_part("stream_mix", spec.streams2) if getattr(spec, "streams2", None) is not None else None
        if spec.arrangement == "streams" and (self.streams is None or (
                spec.feed_forward is not None and (self.norm2 is None or self.streams2 is None))):
            raise ValueError("the streams arrangement needs streams, and norm2 and streams2 for its feed-forward")
        # who reads the stream first in this block, as the block before is told (``then``)
        self.reader = StreamReading(self.streams, self.norm) if spec.arrangement == "streams" else self.norm
        self.reader2 = StreamReading(self.streams2, self.norm2) if spec.arrangement == "streams" and spec.feed_forward is not None else None
        self.mixer = build_part("mixer", spec.mixer)
        if spec.arrangement == "output_norms" and self.norm2 is None and spec.feed_forward is not None:
            raise ValueError("the output_norms arrangement needs norm2 for its feed-forward")
        if spec.feed_forward is None and spec.arrangement not in ("parallel_two_norms", "parallel", "sequential", "output_norms",
                                                                          "norms_around", "streams"):
            raise ValueError(f"the {spec.arrangement} arrangement needs a feed-forward")
        if spec.arrangement == "parallel_two_norms" and spec.feed_forward is not None and self.norm2 is None:
            raise ValueError("the parallel_two_norms arrangement needs norm2 for its feed-forward")
        self.feed_forward = build_part("feed_forward", spec.feed_forward) if spec.feed_forward is not None else None
        if spec.arrangement == "output_norms":
            self.reader = StreamRounding(not getattr(self.mixer, "reads_stream", False))
        self.dtype: Optional[torch.dtype] = None
        self._run = ARRANGEMENTS[spec.arrangement]

    def parts(self) -> Dict[str, Part]:
        out = {"norm": self.norm, "mixer": self.mixer}
        if self.feed_forward is not None:
            out["feed_forward"] = self.feed_forward
        if self.norm2 is not None:
            out["norm2"] = self.norm2
        if self.norm_after is not None:
            out["norm_after"] = self.norm_after
        if self.norm2_after is not None:
            out["norm2_after"] = self.norm2_after
        if self.streams is not None:
            out["streams"] = self.streams
        if self.streams2 is not None:
            out["streams2"] = self.streams2
        return out

    def params(self) -> Dict[str, ParamSpec]:
        """Checkpoint tensor name -> spec, for every tensor of this layer."""
        out = {}
        for part_name, part in self.parts().items():
            for local, pspec in part.params().items():
                key = f"{part_name}.{local}"
                if key not in self.spec.names:
                    raise ValueError(f"the architecture names no tensor for {key!r}")
                out[self.spec.names[key]] = pspec
        return out

    def bind(self, tensors: Dict[str, torch.Tensor], dtype, device) -> None:
        self.dtype = dtype
        for part_name, part in self.parts().items():
            local = {name: tensors[self.spec.names[f"{part_name}.{name}"]] for name in part.params()}
            part.bind(local, dtype, device)

    def forward(self, x: torch.Tensor, batch, cache: LayerCache, normed: Optional[torch.Tensor] = None,
                then: Optional[Part] = None) -> Optional[torch.Tensor]:
        """Updates the fp32 residual ``x`` in place. ``normed``: this block's first norm of ``x``, if the
        block before has computed it; ``then``: the first norm of the block that follows (its ``reader``). Returns that
        norm of the result where the block's last launch computed it, else ``None``. In the ``streams`` arrangement ``x`` is
        ``[n, S, dim]``, and norms are those of what is read of the streams."""
        if not getattr(self._run, "defers", False):
            settle(x, batch)          # (an arrangement that knows nothing of sums left to be added)
        if getattr(self._run, "hands_over", False):
            return self._run(self, x, batch, cache, normed=normed, then=then)
        self._run(self, x, batch, cache)
        return None

    @property
    def narrows(self) -> bool:
        """Whether ``forward_wanted`` can be called."""
        return bool(getattr(self._run, "narrows", False))

    def forward_wanted(self, x: torch.Tensor, batch, cache: LayerCache, wanted, normed: Optional[torch.Tensor] = None,
                       then: Optional[Part] = None):
        """``forward`` where nobody reads the stream behind this block but for the tokens of ``wanted``: ``(their rows of the stream, that norm
        of them or None)``. What the block keeps for later steps it keeps of all tokens."""
        settle(x, batch)
        return self._run(self, x, batch, cache, normed=normed, then=then, wanted=wanted)
