"""Layer norm and convolution of steps of several rows a request, in one kernel and in two: rows on either side of a workgroup's blocks,
portions shorter than the carried inputs, and the carried inputs after each portion."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import plain_suripel as S
from test_suripel_kernels_gpu import DEV, dev, step_ctx

# rows a request brings in three steps (0 rows: it is not there), blocks of 5 and of 8 rows
PORTIONS = [([4], [5], [6]), ([1, 2, 5, 6, 7], [3, 1, 10, 4, 1], [2, 16, 1, 15, 8]), ([9, 3, 1] + [1] * 70, [2, 8, 17] + [1] * 69 + [2], [1, 1, 40] + [2] * 70),
            ([133], [2], [7])]


@pytest.mark.parametrize("E", [4, 252, 2048, 2052, 4096])
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("portions", PORTIONS, ids=lambda p: f"{len(p[0])}x{p[0][0]}")
def test_norm_and_convolution(portions, taps, E):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    B = len(portions[0])
    if B > 8 and E > 2052:
        pytest.skip("many requests at small widths only")
    rng = np.random.default_rng(E + B + taps)
    f32 = lambda a: a.astype(np.float32).astype(np.float64)
    weight = rng.normal(size=E) if taps != 3 else None
    cw, slots = f32(rng.normal(size=(E, taps))), list(rng.permutation(B + 3)[:B])
    states = [torch.zeros((B + 4, taps - 1, E), device=DEV) for _ in range(2)]
    carried, at = np.zeros((B, taps - 1, E)), [0] * B
    for lens in portions:
        ctx = step_ctx(at, lens, slots)
        x = f32(rng.normal(size=(sum(lens), E + 4)) * 2 + 0.3)
        xd = dev(x)[:, :E]
        w = dev(weight) if weight is not None else None
        half = ops.layernorm_conv_rows(xd, w, 1e-5, dev(cw), states[0].clone(), ctx, torch.bfloat16)
        got = ops.layernorm_conv_rows(xd, w, 1e-5, dev(cw), states[0], ctx, torch.float32)
        assert got is not None
        two = ops.causal_conv(ops.layernorm(xd, w, 1e-5, torch.float32), dev(cw), states[1], ctx, torch.float32, residual=True)
        h = S.layer_norm(x[:, :E], f32(weight) if weight is not None else np.ones(E), 1e-5)
        row, want = 0, np.empty_like(h)
        for b, n in enumerate(lens):
            seen = np.concatenate([carried[b], h[row:row + n]])
            want[row:row + n] = h[row:row + n] + sum(cw[:, j] * seen[j:j + n] for j in range(taps))
            carried[b] = seen[len(seen) - (taps - 1):]
            row += n
        # a norm's rounding (2^-24 of values up to 10) through up to four products; the carried inputs are norms
        scale = np.abs(want).max()
        for y in (got, two):
            assert np.abs(y.double().cpu().numpy() - want).max() < 1e-5 * scale
        for st in states:
            assert np.abs(st[torch.tensor(slots, device=DEV)].double().cpu().numpy() - carried).max() < 5e-6 * np.abs(h).max()
            untouched = [i for i in range(B + 4) if i not in slots]
            assert not st[torch.tensor(untouched, device=DEV)].any()
        states[1].copy_(states[0])
        at = [a + n for a, n in zip(at, lens)]
        # two results rounded to bfloat16 from the same 32 bits differ nowhere
        assert torch.equal(half, got.bfloat16())


@pytest.mark.parametrize("taps", [1, 3, 4, 5, 9, 10, 16])
@pytest.mark.parametrize("dtypes", ["float32 float32", "float32 bfloat16", "bfloat16 bfloat16"])
def test_convolution_of_portions(dtypes, taps):
    """Nine taps are the most whose state one block of a request reads; ten go to the kernel that moves states on."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    tu, to = (getattr(torch, d) for d in dtypes.split())
    rng = np.random.default_rng(taps)
    C = 300
    for portions in PORTIONS[1:]:
        B = len(portions[0])
        cw, bias, slots = dev(rng.normal(size=(C, taps))), dev(rng.normal(size=C)), list(rng.permutation(B + 2)[:B])
        state = torch.zeros((B + 3, taps - 1, C), device=DEV, dtype=tu) if taps > 1 else None
        carried, at = np.zeros((B, taps - 1, C)), [0] * B
        for lens in portions:
            ctx = step_ctx(at, lens, slots)
            u = dev(rng.normal(size=(sum(lens), C + 1))).to(tu)[:, :C]
            got = ops.causal_conv(u, cw, state, ctx, to, activation="silu", bias=bias).double().cpu().numpy()
            h, w, bb = u.double().cpu().numpy(), cw.double().cpu().numpy(), bias.double().cpu().numpy()
            row, want = 0, np.empty_like(h)
            for b, n in enumerate(lens):
                seen = np.concatenate([carried[b], h[row:row + n]])
                y = bb + sum(w[:, j] * seen[j:j + n] for j in range(taps))
                want[row:row + n] = y / (1 + np.exp(-y))
                carried[b] = seen[len(seen) - (taps - 1):]
                row += n
            # 32-bit sums of up to 17 terms; a result in bfloat16 is half an ulp off
            assert np.abs(got - want).max() < (1e-5 if to == torch.float32 else 2.0 ** -8) * np.abs(want).max()
            if taps > 1:
                assert np.array_equal(state[torch.tensor(slots, device=DEV)].double().cpu().numpy(), carried)
            at = [a + n for a, n in zip(at, lens)]


def test_more_blocks_than_a_grid_has_rows():
    """Rows in blocks of eight, each of one request, are up to (T + 7 B) / 8: with 21,000 requests of 1 to 40 rows more than 65,535, as with
    600,000 rows of one; the store behind the convolution counts them alike."""
    import torch
    from types import SimpleNamespace
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    C, taps, ps = 4, 4, 64
    rng = np.random.default_rng(5)
    for lens in (rng.integers(1, 41, 21000), np.array([600_000]), np.array([524_281, 3])):
        B, T = len(lens), int(lens.sum())
        assert T + 7 * B > 8 * 65535
        i32 = lambda a: torch.tensor(np.asarray(a, dtype=np.int32), device=DEV)
        cu = np.concatenate([[0], np.cumsum(lens)])
        req = np.repeat(np.arange(B), lens)
        pages = -(-lens // ps)
        table = np.full((B, pages.max()), -1)
        for b, a in enumerate(np.cumsum(pages) - pages):
            table[b, :pages[b]] = np.arange(a, a + pages[b])
        table = i32(table)
        place = i32(np.arange(T) - cu[req])
        ctx = SimpleNamespace(cu_q=i32(cu), slots=i32(np.arange(B)[::-1].copy()), req_of_token=i32(req), starts_dev=i32(np.zeros(B)), positions=place,
                              block_table=lambda g: table, B=B, max_q_len=int(lens.max()))
        u, w = dev(rng.normal(size=(T, C))), dev(rng.normal(size=(C, taps)))
        before = dev(rng.normal(size=(B, taps - 1, C)))
        states = [before.clone(), before.clone()]
        got = ops.causal_conv(u, w, states[0], ctx, torch.float32)
        # rows and carried inputs of all requests one behind the other
        r = torch.tensor(req, device=DEV)
        own = ctx.slots.long()[r]
        want = torch.zeros((T, C), dtype=torch.float64, device=DEV)
        for j in range(taps):
            s = place.long() - (taps - 1) + j
            x = torch.where((s >= 0)[:, None], u[(torch.arange(T, device=DEV) - (taps - 1) + j).clamp(min=0)], before[own, (taps - 1 + s).clamp(max=taps - 2)])
            want += x.double() * w[:, j].double()
        assert float((got.double() - want).abs().max()) < 1e-5 * float(want.abs().max())         # (32-bit sums of four products)
        kc, vc = (torch.zeros((int(pages.sum()), 1, *shape), device=DEV) for shape in ((ps, 1), (1, ps)))
        q = ops.conv_qkv_store(u, w, states[1], kc, vc, ctx, 0, 2, 1, 1, 1, ps, torch.float32)
        assert torch.equal(q, got[:, :2]) and torch.equal(states[0], states[1])
        page, off = table[r, place.long() // ps].long(), place.long() % ps
        assert torch.equal(kc[page, 0, off, 0], got[:, 2]) and torch.equal(vc[page, 0, 0, off], got[:, 3])


@pytest.mark.parametrize("taps", [4, 8, 12, 16])
@pytest.mark.parametrize("C", [5, 256, 1030])
def test_weights_in_pieces_and_number_by_number(taps, C):
    """Weights at a multiple of 16 bytes are read in fours, others one by one: the same sums, so the same bits; and the formula."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(taps * 7 + C)
    lens = [40, 1, 9, 23]                   # (73 rows: long convolutions of fewer than 64 go another way)
    ctx = step_ctx([3] * 4, lens, [2, 0, 3, 1])
    u, w = rng.normal(size=(ctx.T, C)).astype(np.float32), rng.normal(size=(C, taps)).astype(np.float32)
    held = rng.normal(size=(5, taps - 1, C)).astype(np.float32)
    room = torch.empty(C * taps + 1, device=DEV)
    got = []
    for shift in (0, 1):
        wd = room[shift:shift + C * taps].view(C, taps).copy_(torch.tensor(w))
        state = torch.tensor(held, device=DEV)
        got.append((ops.causal_conv(torch.tensor(u, device=DEV), wd, state, ctx, torch.float32).cpu(), state.cpu()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    r = 0
    for n, slot in zip(lens, [2, 0, 3, 1]):
        x = np.concatenate([held[slot], u[r:r + n]]).astype(np.float64)
        want = sum(w[:, j].astype(np.float64) * x[j:j + n] for j in range(taps))
        # 32-bit sums of up to 16 products
        assert np.abs(got[0][0].numpy()[r:r + n] - want).max() < 16 * 2.0 ** -24 * (np.abs(w).astype(np.float64).sum(1) * np.abs(x).max()).max()
        assert np.array_equal(got[0][1].numpy()[slot], x[n:].astype(np.float32))
        r += n
