"""One step's batch: segments of different requests laid end to end.

``StepEntry`` is what a caller hands in: a request, its next tokens (a portion
of its prompt, cut anywhere, or one decoded token) and the places among them
whose logits are wanted.  ``StepContext`` is what the model's parts see: flat
per-token arrays on the device, per-segment arrays, per cache group the block
tables and the slot of every token, plus host copies of the sizes that pick
kernels.
"""
from __future__ import annotations

import dataclasses
from typing import Any, Optional, Sequence

import numpy as np
import torch

from ..ops.transfer import to_device

DECODE_BUCKET = 1024


def decode_bucket(max_context_len: int) -> int:
    return -(-max_context_len // DECODE_BUCKET) * DECODE_BUCKET


@dataclasses.dataclass
class StepEntry:
    rid: Any
    tokens: Sequence[int]
    want: Sequence[int] = ()


@dataclasses.dataclass
class GroupContext:
    block_table: torch.Tensor  # int32 [R, width]
    slot_mapping: torch.Tensor  # int32 [N]
    width: int
    retention: tuple
    seg_lens: list = dataclasses.field(default_factory=list)  # host copies, for kernel work lists
    seg_starts: list = dataclasses.field(default_factory=list)
    meta: dict = dataclasses.field(default_factory=dict)  # kernel launch plans, filled lazily
    # In a step of single tokens only: the context length the kernels' work is laid out for, a multiple of
    # DECODE_BUCKET that no request of the step exceeds.  Grids and key ranges then depend on the number of
    # requests and this bound alone, so a recorded graph of the step fits every step with the same two numbers.
    decode_bucket: Optional[int] = None


@dataclasses.dataclass
class StepContext:
    ops: Any
    dtype: torch.dtype
    device: torch.device
    num_tokens: int
    num_segments: int
    token_ids: torch.Tensor  # int32 [N]
    prev_token_ids: torch.Tensor  # int32 [N]: the token before each token in its sequence, -1 for a first token
    positions: torch.Tensor  # int32 [N]
    token_segment: torch.Tensor  # int32 [N]
    cu_seqlens: torch.Tensor  # int32 [R + 1]
    context_lens: torch.Tensor  # int32 [R]: tokens of the request after this step
    state_slots: torch.Tensor  # int32 [R]
    state_phase: torch.Tensor  # int32 [R]: the half of a two-halved per-request state that this step reads
    logits_indices: torch.Tensor  # int32 [M]
    groups: list[GroupContext]
    # host copies
    seg_lens: list[int]
    seg_starts: list[int]  # position of each segment's first token
    max_seg_len: int
    max_context_len: int
    page_size: int
    every_row: bool = False  # logits_indices is known to be 0, 1, .. N - 1
    # ``tap(part, name, value)``: installed by whoever wants to watch a step (tests, benchmarks).  A part may
    # hand it named intermediate values; if the tap returns something, the part goes on with that instead.
    tap: Optional[Any] = None
    scratch: dict = dataclasses.field(default_factory=dict)


class StepLayout:
    """Where each of a step's arrays lies in ONE flat int32 buffer: per token (ids, positions, segment),
    per segment (bounds, context lengths, state slots), the wanted rows, and per cache group a block table
    ``[segments, width]`` and the slot of every token.  The step function builds such a buffer afresh for
    every step; a recorded step keeps one on the device for good.  Both fill it with :func:`fill_step`
    and make their :class:`StepContext` with :func:`context_over`, so a new per-step array is added in
    these three places and nowhere else."""

    def __init__(self, num_tokens: int, num_segments: int, num_wanted: int, widths: Sequence[int]) -> None:
        N, R = num_tokens, num_segments
        self.num_tokens, self.num_segments, self.num_wanted, self.widths = N, R, num_wanted, list(widths)
        fields = [("token_ids", N), ("prev_token_ids", N), ("positions", N), ("token_segment", N), ("cu_seqlens", R + 1),
                  ("context_lens", R), ("state_slots", R), ("state_phase", R), ("logits_indices", num_wanted)]
        for g, w in enumerate(self.widths):
            fields += [(f"block_table{g}", R * w), (f"slot_mapping{g}", N)]
        self.bounds, o = {}, 0
        for name, n in fields:
            self.bounds[name] = (o, o + n)
            o += n
        self.size = o

    def view(self, flat, name: str):
        lo, hi = self.bounds[name]
        return flat[lo:hi]


def table_widths(cache, entries: Sequence[StepEntry]) -> list:
    """The block tables' widths that this step needs: the longest table of each group."""
    return [max(len(cache.table(e.rid, g.index)) for e in entries) for g in cache.groups]


def fill_step(layout: StepLayout, flat: np.ndarray, cache, entries: Sequence[StepEntry], vocab_size: int,
              stamps: Optional[list] = None, every_row: bool = False):
    """Writes the step's numbers into ``flat`` (int32, ``layout.size`` long).  Every entry's request must
    hold a reservation for ``len(tokens)`` tokens in ``cache``.  ``stamps``: a list with one place per
    segment that the caller keeps between steps over the same buffer; a block-table row is then written
    only if the request in that row, this life of it, or its tables changed since the row was written
    (:meth:`~..cache.manager.CacheManager.table_stamp`).  ``every_row``: every row of a step of single tokens is wanted,
    whatever its entry says.  Returns ``(seg_lens, seg_starts)``."""
    if all(len(e.tokens) == 1 for e in entries) and layout.num_tokens == layout.num_segments == len(entries):
        return _fill_singles(layout, flat, cache, entries, vocab_size, stamps, every_row)
    ps = cache.page_size
    v = lambda name: layout.view(flat, name)
    tok, pos, seg, cu = v("token_ids"), v("positions"), v("token_segment"), v("cu_seqlens")
    ctx_lens, slots, want = v("context_lens"), v("state_slots"), v("logits_indices")
    phase, prev = v("state_phase"), v("prev_token_ids")
    tables = [v(f"block_table{g.index}") for g in cache.groups]
    maps = [v(f"slot_mapping{g.index}") for g in cache.groups]
    seg_lens, seg_starts = [], []
    in_page = np.arange(ps, dtype=np.int32)
    o = w = 0
    cu[0] = 0
    for i, e in enumerate(entries):
        n = len(e.tokens)
        if n < 1:
            raise ValueError("every entry of a step needs at least one token")
        start = cache.num_tokens(e.rid)
        if n == 1:
            t = int(e.tokens[0])
            if not 0 <= t < vocab_size:
                raise ValueError(f"request {e.rid!r}: token id outside 0..{vocab_size - 1}")
            tok[o], pos[o], seg[o] = t, start, i
            prev[o] = cache.last_token(e.rid)
        else:
            t = np.asarray(e.tokens, dtype=np.int64)
            if t.view(np.uint64).max() >= vocab_size:  # (a negative one is a very large one so)
                raise ValueError(f"request {e.rid!r}: token id outside 0..{vocab_size - 1}")
            tok[o: o + n] = t
            prev[o] = cache.last_token(e.rid)
            prev[o + 1: o + n] = t[:-1]
            pos[o: o + n] = np.arange(start, start + n)
            seg[o: o + n] = i
        for x in e.want:
            if not 0 <= x < n:
                raise ValueError(f"request {e.rid!r}: wanted place {x} outside its {n} tokens")
            if w < layout.num_wanted:
                want[w] = o + x
            w += 1
        cu[i + 1] = o + n
        ctx_lens[i], slots[i], phase[i] = start + n, cache.slot(e.rid), cache.state_phase(e.rid)
        stamp = cache.table_stamp(e.rid) if stamps is not None else None
        fresh = stamps is None or stamps[i] != stamp
        for g, width, bt, sm in zip(cache.groups, layout.widths, tables, maps):
            table = cache.table(e.rid, g.index)
            if len(table) > width:
                raise AssertionError(f"request {e.rid!r}: {len(table)} pages in a block table of {width}")
            if fresh:
                row = bt[i * width: (i + 1) * width]
                row[: len(table)] = table
                row[len(table):] = -1
            if n == 1:
                page = table[start // ps] if start // ps < len(table) else -1
                if page < 0:
                    raise AssertionError(f"request {e.rid!r}: a new token has no page in group {g.index}")
                sm[o] = page * ps + start % ps
            else:
                first, last = start // ps, (start + n - 1) // ps
                pages = table[first: last + 1]
                if len(pages) <= last - first or min(pages) < 0:
                    raise AssertionError(f"request {e.rid!r}: a new token has no page in group {g.index}")
                slots_of = np.add.outer(np.array(pages, np.int32) * np.int32(ps), in_page).reshape(-1)
                sm[o: o + n] = slots_of[start - first * ps: start - first * ps + n]
        if stamps is not None:
            stamps[i] = stamp
        seg_lens.append(n)
        seg_starts.append(start)
        o += n
    if o != layout.num_tokens or len(entries) != layout.num_segments:
        raise AssertionError("the entries do not fit the layout they are written into")
    return seg_lens, seg_starts


def _fill_singles(layout: StepLayout, flat: np.ndarray, cache, entries: Sequence[StepEntry], vocab_size: int,
                  stamps: Optional[list], every_row: bool):
    """:func:`fill_step` where every entry has one token.  The device waits for these lines in every decode step, so the
    numbers are gathered in lists and written at once (laying out a step of 64 requests 151 -> 89 us)."""
    ps, groups = cache.page_size, [(g.index, w, layout.view(flat, f"block_table{g.index}"), [])
                                   for g, w in zip(cache.groups, layout.widths)]
    tok, prev, pos, slots, phase, want = [], [], [], [], [], []
    for i, e in enumerate(entries):
        r = cache.requests[e.rid]
        t, start, tables = int(e.tokens[0]), r.num_tokens, r.tables
        if not 0 <= t < vocab_size:
            raise ValueError(f"request {e.rid!r}: token id outside 0..{vocab_size - 1}")
        if not every_row:
            for x in e.want:
                if x != 0:
                    raise ValueError(f"request {e.rid!r}: wanted place {x} outside its 1 tokens")
                want.append(i)
        tok.append(t)
        prev.append(r.last_token)
        pos.append(start)
        slots.append(r.slot)
        phase.append(r.steps & 1)
        fresh = True
        if stamps is not None:
            stamp = (r.serial, *r.versions)
            fresh = stamps[i] != stamp
        at, off = start // ps, start % ps
        for gi, width, bt, sm in groups:
            table = tables[gi]
            if fresh:
                n = len(table)
                if n > width:
                    raise AssertionError(f"request {e.rid!r}: {n} pages in a block table of {width}")
                bt[i * width: i * width + n] = table
                bt[i * width + n: (i + 1) * width] = -1
            page = table[at] if at < len(table) else -1
            if page < 0:
                raise AssertionError(f"request {e.rid!r}: a new token has no page in group {gi}")
            sm.append(page * ps + off)
        if stamps is not None:
            stamps[i] = stamp
    n = len(entries)
    row = list(range(n + 1))
    # (the layout's order: ids, tokens before, positions, segments, bounds, context lengths, slots, phases, wanted rows)
    head = tok + prev + pos + row[:n] + row + [p + 1 for p in pos] + slots + phase + (row[:n] if every_row else want)[: layout.num_wanted]
    flat[: len(head)] = head
    for gi, _, _, sm in groups:
        layout.view(flat, f"slot_mapping{gi}")[:] = sm
    return [1] * n, pos


def context_over(layout: StepLayout, flat: torch.Tensor, cache, ops, dtype, device, *, seg_lens, seg_starts,
                 max_context_len: int, bucket: Optional[int], tap=None, every_row: bool = False) -> StepContext:
    """The :class:`StepContext` whose arrays are views of ``flat`` (on the device the model runs on).
    ``bucket``: see :class:`GroupContext`; ``every_row``: see :class:`StepContext`."""
    R = layout.num_segments
    d = lambda name: layout.view(flat, name)
    groups = []
    for g, width in zip(cache.groups, layout.widths):
        groups.append(GroupContext(block_table=d(f"block_table{g.index}").view(R, width),
                                   slot_mapping=d(f"slot_mapping{g.index}"), width=width, retention=g.retention,
                                   seg_lens=seg_lens, seg_starts=seg_starts, decode_bucket=bucket))
    return StepContext(
        ops=ops, dtype=dtype, device=torch.device(device), num_tokens=layout.num_tokens, num_segments=R,
        token_ids=d("token_ids"), prev_token_ids=d("prev_token_ids"), positions=d("positions"), token_segment=d("token_segment"),
        cu_seqlens=d("cu_seqlens"), context_lens=d("context_lens"), state_slots=d("state_slots"),
        state_phase=d("state_phase"),
        logits_indices=d("logits_indices"), groups=groups, seg_lens=seg_lens, seg_starts=seg_starts,
        max_seg_len=max(seg_lens), max_context_len=max_context_len, page_size=cache.page_size, every_row=every_row, tap=tap)


def build_context(ops, dtype, device, cache, entries: Sequence[StepEntry], vocab_size: int,
                  tap=None) -> StepContext:
    """Lays the entries end to end, in one buffer sent to the device in one copy.  Every entry's request
    must hold a reservation for ``len(tokens)`` tokens in ``cache``."""
    if len(entries) == 0:
        raise ValueError("a step needs at least one entry and every entry at least one token")
    layout = StepLayout(sum(len(e.tokens) for e in entries), len(entries), sum(len(e.want) for e in entries),
                        table_widths(cache, entries))
    flat = np.empty(layout.size, np.int32)
    seg_lens, seg_starts = fill_step(layout, flat, cache, entries, vocab_size)
    host = torch.from_numpy(flat)
    dev = to_device(host, device) if torch.device(device).type != "cpu" else host
    longest = max(s + n for s, n in zip(seg_starts, seg_lens))
    return context_over(layout, dev, cache, ops, dtype, device, seg_lens=seg_lens, seg_starts=seg_starts,
                        max_context_len=longest, bucket=decode_bucket(longest) if max(seg_lens) == 1 else None, tap=tap,
                        every_row=all(len(e.tokens) == 1 and len(e.want) == 1 for e in entries))
