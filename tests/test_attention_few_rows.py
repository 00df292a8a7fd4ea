"""Attention of requests with up to 16 rows a key/value head: the work list on the CPU, the kernel against the plain formula."""
import math

import numpy as np
import pytest
import torch

from xyntetik_runner_amd.engine.batch import Chunked, FEW_MIN_RANGE, few_row_items, first_key


@pytest.mark.parametrize("mask", [None, 40, Chunked(48)])
@pytest.mark.parametrize("extra", [False, True])
@pytest.mark.parametrize("room", [0, 1, 7, 64])
def test_items_cover_every_key_once(mask, extra, room):
    rng = np.random.default_rng(room + 2 * extra)
    starts, lens = rng.integers(0, 700, 9), rng.integers(1, 4, 9)
    starts[0] = 0
    req, q0s = np.arange(9) + 3, np.cumsum(lens) - lens
    items, extras, n_slots = few_row_items(req, starts, lens, q0s, mask, 9 + room, extra, first_slot=5)
    paired = few_row_items(req, starts, lens, q0s, mask, 9 + room, extra, first_slot=5, pair_at=7)[0]
    assert paired[:7].tolist() == items[:7].tolist() and sorted(paired.tolist()) == sorted(items.tolist())
    assert paired[7:].tolist() == (items[7:][::-1] if 7 < len(items) <= 14 else items[7:]).tolist()
    longest = {it[10]: -(-max(x[3] - x[2] for x in items.tolist() if x[10] == it[10]) // 32) for it in items.tolist()}
    assert len(items) <= 9 + room and (np.diff([longest[i] for i in items[:, 10]]) <= 0).all()
    taken = []
    for i in range(9):
        mine = sorted((it for it in items.tolist() if it[0] == req[i]), key=lambda it: it[2])
        at = first_key(mask, int(starts[i])) // 32 * 32
        for it in mine:
            assert it[2] == at and it[3] > at and it[5:8] == [q0s[i], lens[i], starts[i]] and it[10] == i and it[11] == len(mine)
            at = it[3]
        assert at == starts[i] + lens[i]
        slots = [it[4] for it in mine]
        if len(mine) == 1 and not extra:
            assert slots == [-1]
        else:
            assert slots == list(range(mine[0][8], mine[0][8] + len(mine))) and mine[0][9] == len(mine) + extra
            taken += slots + ([int(extras[i, 2])] if extra else [])
            if extra:
                assert extras[i].tolist() == [req[i], 0, slots[-1] + 1, q0s[i], lens[i], starts[i], 0, 0]
    assert sorted(taken) == list(range(5, 5 + n_slots))
    if room == 64 and mask is None:
        assert (items[:, 3] - items[:, 2]).max() <= 32 * max(FEW_MIN_RANGE, -(-int((-(-(starts + lens) // 32)).sum()) // room))


CASES = [
    # H, Hk, D, Dv, page, mask, starts, q_lens
    (4, 1, 32, 32, 32, None, [0, 31, 32, 33], [1, 1, 1, 1]),
    (8, 2, 128, 128, 64, None, [0, 63, 64, 127, 128, 129, 500, 1900], [1] * 8),
    (8, 2, 64, 64, 64, None, [1000, 5, 191, 192, 193], [1, 4, 3, 2, 1]),         # 16, 12, 8 and 4 rows
    (16, 1, 64, 32, 32, None, [300, 2], [1, 1]),                                  # 16 heads a group; values of another size
    (5, 5, 128, 128, 128, 100, [0, 99, 100, 101, 700], [16, 9, 3, 1, 2]),        # a window
    (6, 2, 256, 256, 32, None, [400, 2], [5, 1]),
    (4, 2, 256, 192, 64, Chunked(64), [63, 64, 200], [2, 1, 3]),
    (4, 2, 128, 128, 64, None, [5000], [1]),                                      # more than 64 pages
    (3, 3, 96, 96, 32, 33, [3000, 40], [1, 1]),
]


@pytest.mark.gpu
@pytest.mark.parametrize("room", [1, 1024])
@pytest.mark.parametrize("case", CASES)
def test_few_rows_kernel(case, room, monkeypatch):
    from test_kernels_gpu import DEV, FakeCtx, fill_cache, ref_attention, scatter_pages
    from xyntetik_runner_amd.csrc.ops import load_ops
    from xyntetik_runner_amd.engine import batch
    H, Hk, D, Dv, ps, mask, starts, q_lens = case
    monkeypatch.setattr(batch, "FEW_SLOTS", room)
    torch.manual_seed(D + len(starts))
    lens = [s + n for s, n in zip(starts, q_lens)]
    tables, n_pages = scatter_pages(lens, ps, D)
    ctx = FakeCtx(starts, q_lens, tables, ps)
    ctx.plans_few_rows, ctx._plans, ctx.device = True, {}, DEV
    ctx.attention_plan = lambda *a, **k: batch.StepContext.attention_plan(ctx, *a, **k)
    T = sum(q_lens)
    q = torch.randn(T, H, D).bfloat16()
    k_seq = [torch.randn(n, Hk, D).bfloat16() for n in lens]
    v_seq = [torch.randn(n, Hk, Dv).bfloat16() for n in lens]
    # (a size of its own for values: caches filled apart)
    kc, _ = fill_cache(k_seq, [torch.zeros(n, Hk, D).bfloat16() for n in lens], tables, n_pages, ps, torch.bfloat16)
    _, vc = fill_cache([torch.zeros(n, Hk, Dv).bfloat16() for n in lens], v_seq, tables, n_pages, ps, torch.bfloat16)
    scale = 1 / math.sqrt(D)
    window = mask if isinstance(mask, int) else None
    chunk = mask.size if isinstance(mask, Chunked) else None
    want = torch.empty(T, H, Dv, dtype=torch.float64)
    r = 0
    for b, n in enumerate(q_lens):
        for i in range(n):
            p = starts[b] + i
            lo = first_key(mask, p)
            for h in range(H):
                g = h // (H // Hk)
                s = (k_seq[b][lo:p + 1, g].double() @ q[r, h].double()) * scale
                want[r, h] = torch.softmax(s, 0) @ v_seq[b][lo:p + 1, g].double()
            r += 1
    plan = ctx.attention_plan(0, H // Hk, mask, Hk, ps, few_rows=2 if D + Dv <= 256 else 1)
    assert plan.n_few >= len(starts) and plan.n_items == plan.n_cta_items == plan.n_jobs == 0
    for _ in range(3):          # (the counters are zero again after every launch)
        got = load_ops().attention(q.to(DEV).reshape(T, H * D).contiguous(), kc, vc, ctx, 0, H, Hk, D, ps, scale, window, chunk=chunk, v_head_dim=Dv)
        assert int(plan.counters.abs().sum()) == 0
        got = got.cpu().reshape(T, H, Dv)
        assert torch.isfinite(got.float()).all()
        # probabilities and the result in bfloat16 (2^-9 each of a value) against the largest output
        err = (got.double() - want).abs().amax() / want.abs().amax()
        assert err < 1.2e-2, float(err)


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hk,D,Dv", [(4, 1, 128, 128), (16, 1, 64, 32), (12, 1, 256, 192), (9, 1, 96, 96), (16, 1, 128, 128), (1, 1, 32, 32)])
@pytest.mark.parametrize("least", [1, 3])
def test_many_ranges_added_up(H, Hk, D, Dv, least, monkeypatch):
    """A row block of 1 to 157 key ranges (16, 17, 64, 65 and 128 among them): the last workgroup weighs 64 of them a turn, for one row or sixteen."""
    from xyntetik_runner_amd.engine import batch
    monkeypatch.setattr(batch, "few_row_least", lambda tiles, *a: least)
    starts = [31, 511, 543, 2047, 2079, 4095, 5000]
    test_few_rows_kernel((H, Hk, D, Dv, 64, None, starts, [1] * len(starts)), 1024, monkeypatch)


# What a softmax or a row may have beside its keys; every one of them is in both of the kernel's write-outs.
EXTRAS = {
    "sinks": dict(sinks=True),
    "slopes": dict(slopes=True),
    "slopes in a window, sinks": dict(slopes=True, sinks=True, window=100),
    "cap": dict(cap=1.3),
    "cap and sinks in chunks": dict(cap=1.3, sinks=True, chunk=64),
    "gate": dict(gate=True, scale_out=0.75),
    "gate and sinks in a window": dict(gate=True, scale_out=1.5, sinks=True, window=70),
    "kept keys": dict(window=70, keep=5),
    "kept keys, sinks, slopes, gate": dict(window=40, keep=70, sinks=True, slopes=True, gate=True, scale_out=0.5),
    "kept keys, cap and sinks": dict(window=100, keep=3, sinks=True, cap=1.3),
}


@pytest.mark.gpu
@pytest.mark.parametrize("room", [1, 1024])
@pytest.mark.parametrize("shape", [(8, 2, 64, 64), (4, 1, 128, 64), (5, 5, 32, 32), (2, 1, 256, 128)])
@pytest.mark.parametrize("what", EXTRAS)
def test_few_rows_kernel_with(what, shape, room, monkeypatch):
    """Sinks, distance slopes, a soft cap, gates and kept first keys, one workgroup a request and many; pages that a window has given back are gone."""
    from test_kernels_gpu import DEV, FakeCtx, fill_cache, scatter_pages
    from xyntetik_runner_amd.csrc.ops import load_ops
    from xyntetik_runner_amd.engine import batch
    opt = dict(dict(sinks=False, slopes=False, window=None, chunk=None, keep=0, cap=0.0, gate=False, scale_out=1.0), **EXTRAS[what])
    H, Hk, D, ps = shape
    window, chunk, keep = opt["window"], opt["chunk"], opt["keep"]
    mask = Chunked(chunk) if chunk else window
    monkeypatch.setattr(batch, "FEW_SLOTS", room)
    rng = np.random.default_rng(len(what) * 100 + H + D)
    starts, q_lens = [0, 37, 129, 300, 1500, 64], [1, 2, 1, 2, 1, 1]
    lens = [s + n for s, n in zip(starts, q_lens)]
    tables, n_pages = scatter_pages(lens, ps, D)
    ctx = FakeCtx(starts, q_lens, tables, ps)
    ctx.plans_few_rows, ctx._plans, ctx.device = True, {}, DEV
    ctx.attention_plan = lambda *a, **k: batch.StepContext.attention_plan(ctx, *a, **k)
    bf = lambda a: torch.tensor(a).bfloat16()
    qs = [bf(rng.normal(size=(n, H, D)) * 2) for n in q_lens]
    ks, vs = ([bf(rng.normal(size=(n, Hk, D))) for n in lens] for _ in range(2))
    kc, vc = fill_cache(ks, vs, tables, n_pages, ps, torch.bfloat16)
    if mask:
        tab = ctx._table.cpu()
        for b, s in enumerate(starts):
            tab[b, -(-keep // ps):max(-(-keep // ps), first_key(mask, s) // ps)] = -1
        ctx._table = tab.to(DEV)
    T, scale = sum(q_lens), 1.1 / math.sqrt(D)
    sinks = rng.normal(size=H) * 2
    sinks[0], sinks[-1] = 30.0, -30.0           # one that outweighs every key, one that none feels
    slopes, gate = 2.0 ** -np.linspace(2, 7, H), rng.normal(size=(T, H + 2))
    dev = lambda a: torch.tensor(a, dtype=torch.float32, device=DEV)
    want, r = np.empty((T, H, D)), 0
    for b, n in enumerate(q_lens):
        for i in range(n):
            p = starts[b] + i
            js = np.array(sorted(set(range(min(keep, p + 1))) | set(range(first_key(mask, p), p + 1))))
            for h in range(H):
                s = ks[b][js, h // (H // Hk)].double().numpy() @ qs[b][i, h].double().numpy() * scale
                if opt["cap"]:
                    s = opt["cap"] * np.tanh(s / opt["cap"])
                if opt["slopes"]:
                    s = s - np.float64(np.float32(slopes[h])) * (p - js)
                top = max(s.max(), sinks[h]) if opt["sinks"] else s.max()
                e = np.exp(s - top)
                o = e / (e.sum() + (np.exp(sinks[h] - top) if opt["sinks"] else 0.0)) @ vs[b][js, h // (H // Hk)].double().numpy()
                want[r, h] = o * (1 / (1 + np.exp(-gate[r, h])) if opt["gate"] else 1.0) * opt["scale_out"]
            r += 1
    q = torch.cat(qs).reshape(T, H * D).contiguous().to(DEV)
    more = {**({"extra_slot": True} if keep else {}), "few_rows": 2 if 2 * D <= 256 else 1, "few_channels": 2 * D}
    plan = ctx.attention_plan(0, H // Hk, mask, Hk, ps, **more)
    assert plan.n_few >= len(starts) and plan.n_items == plan.n_cta_items == plan.n_jobs == 0
    for _ in range(2):
        got = load_ops().attention(q, kc, vc, ctx, 0, H, Hk, D, ps, scale, window, chunk=chunk, keep_first=keep, softcap=opt["cap"],
                                   slopes=dev(slopes) if opt["slopes"] else None, sinks=dev(sinks) if opt["sinks"] else None,
                                   gate=dev(gate)[:, :H] if opt["gate"] else None, out_scale=opt["scale_out"]).cpu().double().numpy().reshape(T, H, D)
        assert len(ctx._plans) == 1 and int(plan.counters.abs().sum()) == 0 and np.isfinite(got).all()
        # probabilities and the result in bfloat16 (2^-9 each of a value) against the largest output, as above
        assert np.abs(got - want).max() < 1.2e-2 * np.abs(want).max()


# (tiles, rows, channels of a key and a value): whole, ranges of 3 tiles and more, 16 ranges, 32
@pytest.mark.parametrize("args,least", [((10, 4, 256), 10), ((11, 4, 256), 3), ((13, 16, 256), 13), ((14, 16, 256), 3), ((9, 1, 256), 9), ((10, 1, 256), 3),
                                        ((15, 4, 128), 15), ((16, 4, 128), 3), ((125, 4, 256), 8), ((199, 4, 256), 13), ((200, 4, 256), 7), ((399, 16, 256), 25),
                                        ((400, 16, 256), 13), ((250, 4, 128), 16), ((1, 1, 512), 1)])
def test_shortest_ranges(args, least):
    from xyntetik_runner_amd.engine.batch import few_row_least
    assert few_row_least(*args) == least


@pytest.mark.parametrize("B,n,heads", [(32, 17, 8), (32, 32, 8), (64, 33, 2), (1, 1, 8), (16, 9, 32), (4, 3, 1)])
def test_padded_rows_leave_the_requests_their_ranges(B, n, heads):
    """A recorded batch's list: the rows that pad it have an item each, the requests as many ranges together as fill the kernel's workgroups."""
    from xyntetik_runner_amd.engine.batch import FEW_INTS, FEW_SLOTS
    from xyntetik_runner_amd.engine.graphs import StaticDecodeContext, few_row_room
    room = few_row_room(B, 125, heads)
    ctx = object.__new__(StaticDecodeContext)
    key = (4, None, heads, False, 2, 256)
    ctx.B, ctx._plan_splits = B, {key: room}
    starts = np.zeros(B, dtype=np.int32)
    starts[:n] = 3999 - np.arange(n) * 10
    h = np.full(room * FEW_INTS + B * heads, -7, dtype=np.int32)
    ctx._fill_plan(h, 0, key, starts, n)
    items = h[:room * FEW_INTS].reshape(room, FEW_INTS)
    live = items[items[:, 3] > items[:, 2]]
    assert not h[room * FEW_INTS:].any() and (items[len(live):, 2:4] == 0).all()
    ranges = [int((live[:, 0] == b).sum()) for b in range(B)]
    assert ranges[n:] == [1] * (B - n) and n <= sum(ranges[:n]) <= max(n, FEW_SLOTS // heads)
    if n < FEW_SLOTS // heads:
        assert sum(ranges[:n]) > n          # (not all of them whole)
    assert (live[:, 4] < room).all() and len(set(live[live[:, 4] >= 0, 4].tolist())) == int((live[:, 4] >= 0).sum())
    for b in range(n):
        mine = live[live[:, 0] == b]
        assert mine[:, 2].min() == 0 and mine[:, 3].max() == starts[b] + 1 and (mine[:, 11] == len(mine)).all()
