"""One step's batch as the kernels see it.

A step is a list of entries (request, its next tokens, the places whose logits are
wanted).  All tokens of all entries are laid out one after another ("rows"); per
row the device gets its token id, its position in its request and the index of its
request in this batch; per request and cache group the block table.  One pinned
host buffer carries all of it to the device in a single copy.

The reference has two narrower primitives, n consecutive tokens of one sequence
(src/model.h:667-670) and one token each of up to 8 sequences with
per-column position and cache pointers (src/model.h:796-807,
src/cuda.c:4213-4236); an entry list covers both and their mixtures.
"""
from __future__ import annotations

import math
from dataclasses import dataclass, field
from typing import Hashable, List, Optional, Sequence

import numpy as np
import torch

from ..csrc.ops import Chunked      # (a mask of chunks, as the attention op hands it to a step's plan)


@dataclass
class AttentionPlan:
    """The work list of the MFMA attention kernel for one step, cache group, group size and window.

    ``items [c + n, 8]`` int32 on the device: request, first row of a row block, first key,
    end key, partial slot (-1: the item covers all keys of its block and writes the output),
    the request's first row in the step, its number of tokens, its first position.  The first
    ``n_cta_items`` are blocks of 128 rows that a workgroup takes together (its wave w the rows
    from ``row0 + 32 w``, with partial slot ``slot + w``), the other ``n_items`` blocks of 32
    rows, one wave each.
    ``jobs [m, 7]``: request, first row of 32, first slot, number of slots to merge, the
    distance between them, the request's first row in the step and its number of tokens.
    """
    items: torch.Tensor
    n_items: int
    jobs: Optional[torch.Tensor]
    n_jobs: int
    n_slots: int
    n_cta_items: int = 0
    extras: Optional[torch.Tensor] = None      # [n_extras, 8] (see ``plan_attention``, ``extra_slot``)
    n_extras: int = 0
    few: Optional[torch.Tensor] = None         # [n_few, 12]: blocks of up to 16 rows (see ``few_row_items``)
    n_few: int = 0
    counters: Optional[torch.Tensor] = None    # [row blocks of few rows x key/value heads], zero between launches


def first_key(mask, pos: int) -> int:
    """The first key the query at position ``pos`` reads: ``mask`` None (all), a window's length or a ``Chunked``."""
    if not mask:
        return 0
    if isinstance(mask, Chunked):
        return pos - pos % mask.size
    return max(0, pos - mask + 1)


def mask_reach(mask) -> Optional[int]:
    """The most keys a query reads under ``mask`` (None: all)."""
    if not mask:
        return None
    return mask.size if isinstance(mask, Chunked) else int(mask)


# The first four are the attention kernels' shapes.  The last three are tuning, not limits: they
# say how much work gives every one of an MI355X's 256 compute units a workgroup, measured on the
# 8B shape's attention; on another chip or shape they cost speed, never correctness.
ATTN_ROWS = 32          # query rows (token x head-in-group) per work item
ATTN_TILE = 32          # keys per tile; items begin and end on tile edges
ATTN_CTA_ROWS = 128     # rows of an item that a whole workgroup takes
ATTN_CTA_MIN_ROWS = 64  # a request brings at least this many rows to be served by workgroups
ATTN_STREAM_SLOTS = 256 # workgroups of the streaming kernel that run at a time (one a compute unit)
ATTN_MIN_RANGE = 4      # tiles: the shortest key range worth a workgroup
ATTN_CTA_FILL = 256     # 128-row items (times key/value heads) that give every compute unit one workgroup
FEW_ROWS = 16           # rows of an item of the kernel for few rows (a request's tokens x heads-in-group, at most)
FEW_PAGE = 32           # and the smallest page it takes
FEW_INTS = 12           # numbers of such an item
FEW_MIN_RANGE = 3       # tiles: its shortest key range
FEW_SLOTS = 256         # workgroups of it that a step's requests are cut into: one a compute unit (twice as many cost more than they gain:
                        # 8 requests of 1,000 to 2,000 keys 15.0 us -> 15.9, 16 of 330 9.4 -> 10.6, 32 of 1,000 to 2,000 with heads of 64 22.6 -> 23.3)


def key_ranges(tiles: int, share: float) -> int:
    """Into how many key ranges a 32-row block of ``tiles`` tiles is cut, given its share of
    the workgroups that run at a time.

    Measured on MI355X (batch 1-64, 2k and 8k context): the streaming kernel is fastest with
    one round of workgroups and ranges as long as that allows; a range under 4 tiles costs more
    to start and to merge than to run.
    """
    return max(1, min(int(share), tiles // ATTN_MIN_RANGE))


def plan_attention(starts, q_lens, group_size: int, window, n_kv_heads: int,
                   page_size: int = 64, cta_tiles: Optional[int] = None, extra_slot: bool = False, skip=()):
    """Host side of ``AttentionPlan``: ``(cta_items, items, jobs, n_slots)`` as plain Python ints.

    ``window``: None, a window's length, or a ``Chunked``.  ``skip``: requests that are planned elsewhere.

    ``cta_tiles`` fixes the most tiles a 128-row item may cover (for measurements); by
    default it follows from how many such items the step has.

    ``extra_slot``: every block of 32 rows gets one partial slot more than its key ranges fill,
    for a partial result that another kernel brings (attention over entries that are no keys
    of the cache: a layer's block means), and every item leaves a partial result for the merge.
    A fifth value is then returned: one record ``(request, row0, slot, q0, q_len, start, 0, 0)``
    per block of 32 rows, naming that slot.
    """
    blocks, cta_blocks = [], []
    total_tiles = 0
    q0s, acc = [], 0
    for n in q_lens:
        q0s.append(acc)
        acc += n

    def key_range(s, n, row0, rows):
        tok_lo = row0 // group_size
        tok_hi = min(n - 1, (row0 + rows - 1) // group_size)
        lo = first_key(window, s + tok_lo)
        lo = (lo // ATTN_TILE) * ATTN_TILE
        hi = s + tok_hi + 1
        return lo, hi, -(-(hi - lo) // ATTN_TILE)

    for b, (s, n) in enumerate(zip(starts, q_lens)):
        if b in skip:
            continue
        rows = n * group_size
        if rows >= ATTN_CTA_MIN_ROWS and page_size >= ATTN_TILE:
            for row0 in range(0, rows, ATTN_CTA_ROWS):
                cta_blocks.append((b, row0) + key_range(s, n, row0, ATTN_CTA_ROWS))
            continue
        for row0 in range(0, rows, ATTN_ROWS):
            blk = (b, row0) + key_range(s, n, row0, ATTN_ROWS)
            blocks.append(blk)
            total_tiles += blk[4]
    items, cta_items, jobs, slot = [], [], [], 0
    extras = []
    more = 1 if extra_slot else 0
    # longest first: workgroups are started in list order, and a long item started last
    # would run on alone at the end
    cta_blocks.sort(key=lambda blk: -blk[4])
    blocks.sort(key=lambda blk: -blk[4])

    if cta_blocks:
        chunk = cta_tiles
        if chunk is None:
            # A workgroup (two sets of four waves) fills a compute unit.  Whole blocks when they give
            # at least half the units one each: the merge of split blocks costs more than the units
            # left idle (512 tokens after 4,096, 8 key/value heads: 86 us whole, 86 us in ranges of
            # 32 tiles, 101 us in ranges of 16; 512 tokens from 0: 17 us whole, 26 us split).
            # Fewer blocks are cut into about as many ranges as there are units (128 tokens after
            # 8,000: 145 us whole, 44 us in ranges of 32 tiles, 58 us in ranges of 16).
            if len(cta_blocks) * n_kv_heads >= ATTN_CTA_FILL // 2:
                chunk = 1 << 30
            else:
                work = sum(blk[4] for blk in cta_blocks)
                chunk = max(8, -(-work * n_kv_heads // ATTN_CTA_FILL))
        for b, row0, lo, hi, tiles in cta_blocks:
            parts = -(-tiles // chunk)
            if parts <= 1 and not extra_slot:
                cta_items.append((b, row0, lo, hi, -1, q0s[b], q_lens[b], starts[b]))
                continue
            parts = max(1, parts)
            per = -(-tiles // parts)
            first = slot
            k = lo
            while k < hi:
                e = min(hi, k + per * ATTN_TILE)
                cta_items.append((b, row0, k, e, slot, q0s[b], q_lens[b], starts[b]))
                slot += ATTN_CTA_ROWS // ATTN_ROWS
                k = e
            n_parts = (slot - first) // (ATTN_CTA_ROWS // ATTN_ROWS)
            rows = q_lens[b] * group_size
            for w in range(ATTN_CTA_ROWS // ATTN_ROWS):
                if row0 + w * ATTN_ROWS < rows:
                    jobs.append((b, row0 + w * ATTN_ROWS, first + w, n_parts + more, ATTN_CTA_ROWS // ATTN_ROWS, q0s[b], q_lens[b]))
                    if extra_slot:
                        extras.append((b, row0 + w * ATTN_ROWS, slot + w, q0s[b], q_lens[b], starts[b], 0, 0))
            if extra_slot:
                slot += ATTN_CTA_ROWS // ATTN_ROWS

    budget = max(1, ATTN_STREAM_SLOTS // n_kv_heads)       # items that run at a time
    for b, row0, lo, hi, tiles in blocks:
        parts = 1 if len(blocks) >= budget else key_ranges(tiles, budget * tiles / total_tiles)
        if parts <= 1 and not extra_slot:
            items.append((b, row0, lo, hi, -1, q0s[b], q_lens[b], starts[b]))
            continue
        parts = max(1, parts)
        per = -(-tiles // parts)
        first = slot
        k = lo
        while k < hi:
            e = min(hi, k + per * ATTN_TILE)
            items.append((b, row0, k, e, slot, q0s[b], q_lens[b], starts[b]))
            slot += 1
            k = e
        jobs.append((b, row0, first, slot - first + more, 1, q0s[b], q_lens[b]))
        if extra_slot:
            extras.append((b, row0, slot, q0s[b], q_lens[b], starts[b], 0, 0))
            slot += 1
    if extra_slot:
        return cta_items, items, jobs, slot, extras
    return cta_items, items, jobs, slot


def few_row_least(tiles: int, rows: int, channels: int = 256) -> int:
    """Tiles of the shortest key range that pays where the longest request of a step has ``tiles`` tiles, ``rows`` rows a key/value head and ``channels`` of a
    key and its value together.

    The last workgroup of a row block adds the ranges up, in a round of trips to memory for 16 of them (more where there are many rows of many channels, or more ranges): 2 to 3
    us, in which a workgroup goes through 5 tiles of 256 channels, through more of fewer.  Whole and in 2, 4 and 8 ranges, us: 4 x 4 heads of 128, 9 tiles 7.4, 9.1, 8.1;
    12 tiles 8.8, 9.1, 8.8; 16 tiles 10.3, 10.1, 8.8, 7.3; 4 x 16 heads, 12 tiles 9.9, 11.0, 10.2; 16 tiles 11.5, 11.8, 10.8, 9.2; 4 x 4 of 64, 16 tiles 6.9, 8.2, 7.5, 6.5.
    16 ranges and 32: 125 tiles of 4 x 4 heads of 128 9.9 and 10.8, of 4 x 16 13.0 and 14.5; 250 tiles 13.4 and 12.2, 16.2 and 15.9; of 4 x 4 of 64 9.6 and 9.9.  Over 972 pairs of
    heads, requests and tiles 1% to 3% over the best of nine numbers of ranges, none slower than the streaming kernel and its merge."""
    if tiles < (10 + rows // 4) * math.sqrt(256 / channels):
        return tiles
    most = 16 if tiles * channels < (51200 if rows <= 8 else 102400) else 32
    return max(FEW_MIN_RANGE, -(-tiles // most))


def few_row_items(req, starts, lens, q0s, mask, room: int, extra_slot: bool, first_slot: int = 0, pair_at: int = 0, least=None):
    """The work of the kernel for few rows: requests ``req`` of a step, each with one row block (its ``lens[i]`` tokens from row
    ``q0s[i]`` and position ``starts[i]`` on), cut into at most ``room`` key ranges of about one length, so that a
    long request takes as many workgroups as its keys are worth: ``(items [n, 12], extras [len(req), 8], slots)`` as int64 arrays.

    An item: request, 0, first key, end key, partial slot (-1: all its keys), the request's first row, its tokens, its first
    position, the row block's first slot, its slots, its counter and how many items it has.  With ``extra_slot`` a row block has
    one slot more, its last, for a partial result of another kernel (``extras`` as ``plan_attention`` makes them).  ``least``: the tiles of the
    shortest range, from those of the longest request.

    The requests with the longest ranges come first, workgroups start in the items' order.  ``pair_at``: the items that give every compute unit one workgroup, where
    it holds two at a time: if there are up to twice as many, all run at once, and the second half comes shortest first, so that
    a unit has a long and a short one (64 requests of 950 to 1,900 keys 71.3 us -> 68.8, of 100 to 4,000 117.8 -> 96.8; 48 of 950 to 1,900 65.6 -> 57.8)."""
    starts, lens = np.asarray(starts, dtype=np.int64), np.asarray(lens, dtype=np.int64)
    n = len(starts)
    hi = starts + lens
    if mask:
        lo = starts - starts % mask.size if isinstance(mask, Chunked) else np.maximum(0, starts - mask + 1)
        lo = lo // ATTN_TILE * ATTN_TILE
    else:
        lo = 0
    tiles = (hi - lo + (ATTN_TILE - 1)) // ATTN_TILE
    # the shortest length c with at most ``room`` ranges: ceil(t / c) a request, which c >= total / (room - requests) has in any case
    t = tiles.tolist()
    longest = max(t)
    if room > n:
        total = sum(t)
        least = FEW_MIN_RANGE if least is None else max(1, least(longest))
        most = max(least, -(-total // (room - n)))
        for c in range(max(least, -(-total // room)), most, max(1, most // 32)):
            if sum([-(-x // c) for x in t]) <= room:
                most = c
                break
        longest = min(longest, most)
    rec = np.zeros((n, FEW_INTS), dtype=np.int64)            # a request's items have this in common; 1: the keys of a range
    rec[:, 0], rec[:, 2], rec[:, 3], rec[:, 5], rec[:, 6], rec[:, 7], rec[:, 10] = req, lo, hi, q0s, lens, starts, np.arange(n)
    n_slots, extras = 0, rec[:0, :8]
    if longest < max(t) or extra_slot:
        parts = (tiles + (longest - 1)) // longest
        per = (tiles + (parts - 1)) // parts
        parts = (tiles + (per - 1)) // per
        slots = parts + 1 if extra_slot else np.where(parts > 1, parts, 0)
        end = np.cumsum(slots)
        n_slots = int(end[-1])
        rec[:, 1], rec[:, 8], rec[:, 9], rec[:, 11] = per * ATTN_TILE, first_slot + end - slots, slots, parts
        if extra_slot:
            extras = np.zeros((n, 8), dtype=np.int64)
            extras[:, 0], extras[:, 2], extras[:, 3], extras[:, 4], extras[:, 5] = req, rec[:, 8] + parts, q0s, lens, starts
        order = np.argsort(-per, kind="stable")
        parts = parts[order]
        items = np.repeat(rec[order], parts, axis=0)
        k = np.arange(len(items)) - np.repeat(np.cumsum(parts) - parts, parts)
        items[:, 2] += k * items[:, 1]
        items[:, 3] = np.minimum(items[:, 3], items[:, 2] + items[:, 1])
        items[:, 4] = np.where(items[:, 9] > 0, items[:, 8] + k, -1)
        items[:, 1] = 0
    else:
        rec[:, 4], rec[:, 11] = -1, 1
        items = rec[np.argsort(-tiles, kind="stable")]
    if 0 < pair_at < len(items) <= 2 * pair_at:
        items[pair_at:] = items[pair_at:][::-1].copy()
    return items, extras, n_slots


@dataclass
class StepEntry:
    req_id: Hashable
    tokens: Sequence[int]
    want: Sequence[int] = ()        # indices into ``tokens`` whose logits are wanted


class StepContext:
    """Device views of one step's metadata, handed to every part."""

    plans_few_rows = True       # its attention plans know the kernel for few rows
    knows_lengths = True        # ``max_seq_len`` is this step's (a recorded step's lengths change from replay to replay)

    def __init__(self, ops, device, entries: List[StepEntry], request_caches, n_groups: int, pad_to: int = 0):
        self.ops = ops
        self.device = device
        self.entries = entries
        B = len(entries)
        q_lens = [len(e.tokens) for e in entries]
        T = sum(q_lens)
        self.B, self.T = B, T
        self.q_lens = q_lens
        self.starts = [rc.n_tokens for rc in request_caches]            # position of each entry's first token
        self.seq_lens = [s + n for s, n in zip(self.starts, q_lens)]    # length after this step
        self.max_q_len = max(q_lens) if q_lens else 0
        self.max_seq_len = max(self.seq_lens) if B else 0
        nb = [max((len(rc.tables[g]) for rc in request_caches), default=0) for g in range(n_groups)]
        self.table_width = [max(1, w) for w in nb]
        want_rows: List[int] = []
        row0 = 0
        for e, n in zip(entries, q_lens):
            for w in e.want:
                if not (0 <= w < n):
                    raise ValueError(f"request {e.req_id!r}: wanted place {w} is outside its {n} tokens")
                want_rows.append(row0 + w)
            row0 += n
        self.n_want = len(want_rows)

        # ---- pack: [token_ids T][positions T][req_of_token T][cu_q B+1][seq_lens B][slots B][fresh B]
        #            [want W][table g: B * width_g]...
        sizes = [T, T, T, B + 1, B, B, B + B, self.n_want] + [B * w for w in self.table_width]
        offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
        total = int(offs[-1])
        host = torch.empty((max(total, 1),), dtype=torch.int32, pin_memory=True)
        h = host.numpy()
        tok, pos, rot = h[offs[0]:offs[1]], h[offs[1]:offs[2]], h[offs[2]:offs[3]]
        cu = h[offs[3]:offs[4]]
        cu[0] = 0
        r = 0
        for b, (e, n) in enumerate(zip(entries, q_lens)):
            tok[r:r + n] = np.asarray(e.tokens, dtype=np.int64).astype(np.int32)
            pos[r:r + n] = np.arange(self.starts[b], self.starts[b] + n, dtype=np.int32)
            rot[r:r + n] = b
            r += n
            cu[b + 1] = r
        h[offs[4]:offs[5]] = self.seq_lens
        h[offs[5]:offs[6]] = [rc.slot for rc in request_caches]
        h[offs[6]:offs[6] + B] = [1 if rc.fresh else 0 for rc in request_caches]
        h[offs[6] + B:offs[7]] = self.starts
        h[offs[7]:offs[8]] = want_rows
        for g in range(n_groups):
            w = self.table_width[g]
            tab = h[offs[8 + g]:offs[9 + g]].reshape(B, w)
            tab[:] = -1
            for b, rc in enumerate(request_caches):
                t = rc.tables[g]
                tab[b, :len(t)] = t
        dev = host.to(device, non_blocking=True)
        self._host = host      # keep the pinned buffer alive until the copy has run
        self.token_ids = dev[offs[0]:offs[1]]
        self.positions = dev[offs[1]:offs[2]]
        self.req_of_token = dev[offs[2]:offs[3]]
        self.cu_q = dev[offs[3]:offs[4]]
        self.seq_lens_dev = dev[offs[4]:offs[5]]
        self.slots = dev[offs[5]:offs[6]]
        self.fresh = dev[offs[6]:offs[6] + B]
        self.starts_dev = dev[offs[6] + B:offs[7]]
        self.want_rows = dev[offs[7]:offs[8]]
        self._tables = [dev[offs[8 + g]:offs[9 + g]].view(B, self.table_width[g]) for g in range(n_groups)]
        self.fresh_slots_host = [rc.slot for rc in request_caches if rc.fresh]
        self.slots_host = [rc.slot for rc in request_caches]
        self._plans = {}
        self.shared = {}        # what parts make once a step and share between layers (a rotation's table)

    def attention_plan(self, group: int, group_size: int, window, n_kv_heads: int,
                       page_size: int = 64, extra_slot: bool = False, few_rows: int = 0, few_channels: int = 256) -> AttentionPlan:
        """The MFMA attention work list, made once per step and shared by all layers that can.  ``few_rows`` > 0:
        requests of up to 16 rows a key/value head go to the kernel for few rows (where the page size allows), of which a compute unit
        holds so many workgroups; ``few_channels``: those of a key and its value together."""
        key = (group_size, window, n_kv_heads, page_size, extra_slot, few_rows, few_channels)
        plan = self._plans.get(key)
        if plan is None:
            few = [b for b, n in enumerate(self.q_lens) if few_rows and page_size >= FEW_PAGE and n * group_size <= FEW_ROWS]
            planned = plan_attention(self.starts, self.q_lens, group_size, window, n_kv_heads, page_size,
                                     extra_slot=extra_slot, skip=frozenset(few))
            cta_items, items, jobs, n_slots = planned[:4]
            extras = [tuple(x) for x in planned[4]] if extra_slot else []
            flat = [v for it in cta_items + items for v in it] + [v for j in jobs for v in j]
            n_few = n_count = 0
            if few:
                q0s = np.concatenate([[0], np.cumsum(self.q_lens)])[few]
                room = max(len(few), FEW_SLOTS // n_kv_heads)
                few_items, few_extras, more = few_row_items(few, [self.starts[b] for b in few], [self.q_lens[b] for b in few], q0s,
                                                            window, room, extra_slot, n_slots, ATTN_STREAM_SLOTS // n_kv_heads if few_rows == 2 else 0,
                                                            least=lambda t: few_row_least(t, group_size * max(self.q_lens[b] for b in few), few_channels))
                n_slots += more
                n_few, n_count = len(few_items), len(few) * n_kv_heads
                extras += few_extras.tolist()
            flat += [v for x in extras for v in x]
            if few:
                flat += few_items.ravel().tolist() + [0] * n_count
            host = torch.tensor(flat, dtype=torch.int32).pin_memory()
            dev = host.to(self.device, non_blocking=True)
            nc, ni, nj = len(cta_items), len(items), len(jobs)
            nw = (nc + ni) * 8
            nx = nw + nj * 7
            nf = nx + len(extras) * 8
            plan = AttentionPlan(dev[:nw], ni, dev[nw:nx] if nj else None, nj, n_slots, nc,
                                 dev[nx:nf] if extras else None, len(extras),
                                 dev[nf:nf + n_few * FEW_INTS] if n_few else None, n_few, dev[nf + n_few * FEW_INTS:] if n_few else None)
            plan._host = host
            self._plans[key] = plan
        return plan

    def block_table(self, group: int) -> torch.Tensor:
        """``[B, width]`` int32: page of each block of each request of this step, -1 where none."""
        return self._tables[group]
