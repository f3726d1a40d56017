"""The packed batch of one step as the parts see it, and the scratch memory they share."""

from __future__ import annotations

from dataclasses import dataclass, field, replace
from typing import Dict, Optional, Tuple

import torch


class Workspace:
    """Named scratch tensors that live as long as the engine.

    ``get(name, shape, dtype)`` returns a view of a persistent buffer, grown on demand;
    the same name gives the same memory in every step, so a captured HIP graph can be
    replayed. ``freeze()`` forbids further growth (addresses must not change any more).
    """

    def __init__(self, device: torch.device) -> None:
        self.device = device
        self._buffers: Dict[Tuple[str, torch.dtype], torch.Tensor] = {}
        self._frozen = False

    def freeze(self) -> None:
        self._frozen = True

    def get(self, name: str, shape: Tuple[int, ...], dtype: torch.dtype) -> torch.Tensor:
        count = 1
        for s in shape:
            count *= int(s)
        key = (name, dtype)
        buf = self._buffers.get(key)
        if buf is None or buf.numel() < count:
            if self._frozen:
                raise RuntimeError(f"workspace {name!r} would have to grow to {count} elements after freeze()")
            buf = torch.empty(max(count, 1), dtype=dtype, device=self.device)
            self._buffers[key] = buf
        return buf[:count].view(*shape)

    def bytes(self) -> int:
        return sum(b.numel() * b.element_size() for b in self._buffers.values())


@dataclass
class GroupBatch:
    """Per cache group: where this step's tokens live and what they may read."""

    block_table: torch.Tensor           # int32 [rows, max_pages]
    slots: torch.Tensor                 # int32 [tokens]: page * page_size + offset
    kv_lo: Optional[torch.Tensor]       # int32 [tokens] first visible key, or None for 0
    page_size: int = 0


@dataclass
class StepBatch:
    """One step: ``n_tokens`` packed tokens of ``n_rows`` requests, on the device.

    Token ``t`` belongs to row ``token_row[t]``, stands at ``positions[t]`` and sees the
    keys ``[kv_lo[t], kv_hi[t])`` of its row. ``row_slot[r]`` is the request's slot in the
    per-request state tensors. ``logit_rows`` names the tokens whose logits are wanted.
    """

    n_tokens: int
    n_rows: int
    token_ids: torch.Tensor             # int32 [tokens], -1 where an embedding is given
    positions: torch.Tensor             # int32 [tokens]: the token's place in its sequence (and in the cache)
    token_row: torch.Tensor             # int32 [tokens]
    kv_hi: torch.Tensor                 # int32 [tokens]
    row_slot: torch.Tensor              # int32 [rows]
    cu_q: torch.Tensor                  # int32 [rows + 1]
    kv_len: torch.Tensor                # int32 [rows]: keys held after this step
    logit_rows: torch.Tensor            # int32 [wanted]
    logit_slot: torch.Tensor            # int32 [wanted]: the slot of the request a row of logits belongs to (-1: a padding row)
    groups: Dict[int, GroupBatch]
    workspace: Workspace
    # per size of block that a mixer's kernel asked for: (int32 [blocks] row of each block of that
    # many queries of one row, int32 [blocks] its first token), the blocks that see the most keys first
    query_blocks: Dict[int, Tuple[torch.Tensor, torch.Tensor]] = field(default_factory=dict)
    # (int32 [runs] first token, int32 [runs] count): the tokens cut into runs that fill one page of their row in
    # order, and runs of up to a page's worth of other tokens (for the kernels that write the cache by pages)
    page_runs: Optional[Tuple[torch.Tensor, torch.Tensor]] = None
    # int32 [tokens, axes] where a position encoding of the model takes more than one number per token
    position_axes: Optional[torch.Tensor] = None
    pending: Optional[torch.Tensor] = None        # int32 device table: an id <= -2 stands for pending[-2 - id]
    given_embeds: Optional[torch.Tensor] = None   # [m, dim]
    given_rows: Optional[torch.Tensor] = None     # int32 [m] token indices they go to
    # facts known on the host, for choosing kernels
    max_q: int = 1
    max_kv: int = 1
    decode_only: bool = False
    causal_only: bool = True            # no token sees past its own position
    wants_every_token: bool = False     # ``logit_rows`` is 0, 1, ..., n_tokens - 1: every token's logits, in order
    whole_last: bool = False            # every token through the last layer, whichever are wanted (a warm-up: scratch of any step)
    host: dict = field(default_factory=dict)

    def wanted_alone(self) -> Optional["WantedTokens"]:
        """The tokens whose logits are wanted as a step of their own, where that pays (``WantedTokens``)."""
        return WantedTokens(self) if not self.whole_last and WantedTokens.pays(self) else None


class WantedTokens:
    """The tokens of a step whose logits are wanted, as a step of its own: what is left to do behind the last kernel that reads a
    token's row for another token's sake (the last layer's keys, values and states).

    ``batch`` lists them as single tokens, in the order of the logits, that read their requests' caches and write nothing. Its columns, and whatever a
    part hands over on the way, are picked out of the step by ``gather``, the columns by its first call."""

    # Most wanted tokens, and tokens of the step to each of them: attention over single tokens reads a request's keys once for each of them. And the fewest
    # tokens of a step: up to 16 a layer is three launches that wait for its weights, whichever rows they are for.
    MOST, SHARE, TOKENS = 64, 2, 17

    @classmethod
    def pays(cls, batch: "StepBatch") -> bool:
        wanted = int(batch.logit_rows.numel())
        return not batch.decode_only and batch.n_tokens >= cls.TOKENS and wanted <= cls.MOST and wanted * cls.SHARE <= batch.n_tokens

    def __init__(self, batch: "StepBatch") -> None:
        self.rows = batch.logit_rows
        self.count = int(self.rows.numel())
        self._workspace = batch.workspace
        self._columns = []

        def column(name: str, source: torch.Tensor) -> torch.Tensor:
            own = self.buffer(name, source)
            self._columns.append((source, own))
            return own

        groups = {key: replace(g, slots=g.slots[:0], kv_lo=None if g.kv_lo is None else column(f"kv_lo{key}", g.kv_lo))
                  for key, g in batch.groups.items()}
        self.batch = replace(
            batch, n_tokens=self.count, n_rows=self.count, token_ids=batch.token_ids[:0], positions=column("positions", batch.positions),
            token_row=column("token_row", batch.token_row), kv_hi=column("kv_hi", batch.kv_hi), row_slot=batch.row_slot[:0], cu_q=batch.cu_q[:0],
            kv_len=batch.kv_len[:0], groups=groups, query_blocks={}, page_runs=None, position_axes=None, given_embeds=None, given_rows=None, max_q=1,
            decode_only=True, wants_every_token=True, host={})

    def buffer(self, name: str, like: torch.Tensor) -> torch.Tensor:
        """Scratch for the wanted rows of ``like``."""
        return self._workspace.get("wanted." + name, (self.count, *like.shape[1:]), like.dtype)

    def gather(self, *pairs) -> None:
        """``dst[i] = src[rows[i]]`` for every ``(src, dst)``."""
        from ..ops import core

        core.gather_rows(self.rows, [*self._columns, *pairs])
        self._columns = []

    def take(self, name: str, source: torch.Tensor, *pairs) -> torch.Tensor:
        """The wanted rows of ``source`` in scratch memory, and ``pairs`` besides."""
        own = self.buffer(name, source)
        self.gather((source, own), *pairs)
        return own
