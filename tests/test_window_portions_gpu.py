"""Portions on their way through windowed attention: the convolution that stores, queries and keys turned in one kernel, means of blocks eight
positions at a time, and steps that no block's mean can reach; each against the kernels that it stands for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_suripel_kernels_gpu import DEV, dev, step_ctx


def tables_for(B, pages):
    perm = np.random.default_rng(B * 100 + pages).permutation(B * pages)
    return [[int(x) for x in perm[b * pages:(b + 1) * pages]] for b in range(B)]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("H,Hk,D,Dv,taps,ps", [(3, 1, 7, 5, 2, 4), (2, 2, 48, 96, 9, 16), (8, 2, 128, 128, 4, 64), (4, 0, 64, 64, 3, 64)])
def test_convolution_of_portions_and_store(H, Hk, D, Dv, taps, ps, dtype):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dt = load_ops(), getattr(torch, dtype)
    rng = np.random.default_rng(D + taps)
    B, Q, K = 3, H * D, Hk * D
    C = Q + Hk * (D + Dv)
    w, slots, tables = dev(rng.normal(size=(C, taps))), [2, 0, 3], tables_for(B, -(-64 // ps))
    mk = lambda: (torch.zeros((5, taps - 1, C), device=DEV), torch.zeros((B * len(tables[0]), max(Hk, 1), ps, D), dtype=dt, device=DEV),
                  torch.zeros((B * len(tables[0]), max(Hk, 1), Dv, ps), dtype=dt, device=DEV))
    one, two, at = mk(), mk(), [0] * B
    # blocks of 8 that begin on a multiple of 8 and that do not, portions shorter than the carried inputs
    for lens in ([8, 16, 3], [1, 8, 13], [9, 7, 24], [2, 1, 8]):
        ctx = step_ctx(at, lens, slots, [tables])
        u = dev(rng.normal(size=(sum(lens), C + 3)))[:, :C]
        got = ops.conv_qkv_store(u, w, one[0], one[1] if Hk else None, one[2] if Hk else None, ctx, 0, H, Hk, D, Dv, ps, dt)
        y = ops.causal_conv(u, w, two[0], ctx, torch.float32)
        want = ops.qkv_store(y[:, :Q], y[:, Q:Q + K] if Hk else None, y[:, Q + K:] if Hk else None, two[1], two[2], ctx, 0, H, Hk, D, Dv, ps, dt)
        assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(one, two))
        at = [a + n for a, n in zip(at, lens)]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("off", [1, 2, 4])
def test_convolution_and_store_to_values_at_any_address(off, dtype):
    """A value's eight places are stored one by one where the cache is not 16-byte aligned."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dt = load_ops(), getattr(torch, dtype)
    H, Hk, D, ps, taps, lens = 2, 1, 8, 16, 4, [24, 9]
    rng = np.random.default_rng(off)
    C = (H + 2 * Hk) * D
    u, w, tables = dev(rng.normal(size=(sum(lens), C))), dev(rng.normal(size=(C, taps))), tables_for(2, 2)
    ctx = step_ctx([0, 0], lens, [1, 0], [tables])
    got = []
    for at in (0, off):
        kc = torch.zeros((4, Hk, ps, D), dtype=dt, device=DEV)
        vc = torch.zeros((4 * Hk * D * ps + at,), dtype=dt, device=DEV)[at:].view(4, Hk, D, ps)
        got.append((ops.conv_qkv_store(u, w, torch.zeros((3, taps - 1, C), device=DEV), kc, vc, ctx, 0, H, Hk, D, D, ps, dt), kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and bool(got[0][2].any())


@pytest.mark.parametrize("heads,D,rot", [(1, 6, 4), (3, 64, 64), (32, 128, 96), (5, 130, 130), (2, 16, 0)])
def test_queries_and_keys_turned_together(heads, D, rot):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(heads + D)
    T, N = 37, heads * D
    row = dev(rng.normal(size=(T, 2 * N + 3)))
    other = row.clone()
    pos = torch.tensor(rng.integers(0, 5000, size=T), dtype=torch.int32, device=DEV)
    inv = dev(1e4 ** (-np.arange(rot // 2) / max(1, rot // 2))) if rot else None
    ops.rotate_pair_(row[:, :N], row[:, N:2 * N], pos, inv, heads, D, rot, 1.0, 0.25)
    ops.rotate_rows_(other[:, :N], pos, inv, heads, D, rot, 1.0)
    ops.rotate_rows_(other[:, N:2 * N], pos, inv, heads, D, rot, 0.25)
    # (two products and a sum, fused or not: 2^-23 of numbers up to 8)
    assert float((row - other).abs().max()) <= 8 * 2.0 ** -23 and torch.equal(row[:, 2 * N:], other[:, 2 * N:])


@pytest.mark.parametrize("P,ps", [(8, 16), (64, 64), (24, 32), (12, 16), (64, 32)])
def test_means_of_blocks(P, ps):
    """Sums of up to 64 values in 32 bits, rounded to bfloat16: half an ulp, or one where a sum's own rounding decides."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(P)
    B, Hk, D, Dv, pages = 2, 2, 32, 48, 256 // ps
    tables = tables_for(B, pages)
    kc = dev(rng.normal(size=(B * pages, Hk, ps, D))).bfloat16()
    vc = dev(rng.normal(size=(B * pages, Hk, Dv, ps))).bfloat16()
    pk, pv = torch.zeros_like(kc), torch.zeros_like(vc)
    starts, lens = [P - 1, 0], [200 - P, 131]
    ops.pool_blocks(pk, pv, kc, vc, step_ctx(starts, lens, [0, 1], [tables, tables]), 0, 1, Hk, D, Dv, P, ps)
    for b in range(B):
        keys = torch.cat([kc[p].double() for p in tables[b]], dim=1)                     # [Hk, positions, D]
        vals = torch.cat([vc[p].double() for p in tables[b]], dim=2)
        for blk in range(pages * ps // P):
            done = starts[b] // P <= blk < (starts[b] + lens[b]) // P
            page, off = tables[b][blk // ps], blk % ps
            want_k = keys[:, blk * P:(blk + 1) * P].mean(dim=1) if done else torch.zeros_like(keys[:, 0])
            want_v = vals[:, :, blk * P:(blk + 1) * P].mean(dim=2) if done else torch.zeros_like(vals[:, :, 0])
            for got, want in ((pk[page, :, off], want_k), (pv[page, :, :, off], want_v)):
                assert float((got.double() - want).abs().max()) <= 2.0 ** -8 * max(1e-6, float(want.abs().max())) * 1.01, (b, blk)


@pytest.mark.parametrize("G", [1, 4])
@pytest.mark.parametrize("longest", [40, 95, 96, 97, 130])
def test_steps_that_no_mean_reaches(longest, G):
    """Window 80, blocks of 16: the first mean is read at position 95 (a length of 96)."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(longest)
    B, Hk, D, ps, size, P = 2, 2, 64, 32, 80, 16
    H, pages = Hk * G, 6
    tables = tables_for(B, pages)
    kc = dev(rng.normal(size=(B * pages, Hk, ps, D))).bfloat16()
    vc = dev(rng.normal(size=(B * pages, Hk, D, ps))).bfloat16()
    pk, pv = torch.zeros_like(kc), torch.zeros_like(vc)
    lens = [longest - 3, 7]
    ctx = step_ctx([3, 0], lens, [0, 1], [tables, tables])
    ops.pool_blocks(pk, pv, kc, vc, step_ctx([0, 0], [longest, 7], [0, 1], [tables, tables]), 0, 1, Hk, D, D, P, ps)
    q = dev(rng.normal(size=(sum(lens), H * D))).bfloat16()
    args = (q, kc, vc, pk, pv, ctx, 0, 1, H, Hk, D, D, ps, D ** -0.5, size, P)
    got = ops.attention_pooled(*args)
    ctx.knows_lengths = False
    with_slot = ops.attention_pooled(*args)
    plain = ops.attention_pooled(*args, matrix_cores=False)
    # probabilities in bfloat16 (2^-9 of each) and the result's rounding
    for other in (with_slot, plain):
        assert float((got.double() - other.double()).abs().max()) <= 2.0 ** -6 * float(plain.abs().max())


@pytest.mark.parametrize("T,H,Dv", [(1, 1, 128), (3, 3, 128), (37, 5, 128), (8, 4, 132), (129, 3, 256)])
@pytest.mark.parametrize("gate_first", [False, True])
def test_gated_norm_of_two_heads_a_wave(T, H, Dv, gate_first):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(T + Dv)
    o, gate, w = dev(rng.normal(size=(T, H * Dv))), dev(rng.normal(size=(T, H * Dv + 4)))[:, :H * Dv], dev(rng.normal(size=Dv))
    got = ops.gated_rmsnorm(o, gate, w, H, Dv, 1e-5, torch.bfloat16, gate_first=gate_first)
    x, g = o.double().view(T, H, Dv), gate.double().reshape(T, H, Dv)
    g = g * torch.sigmoid(g)
    x = x * g if gate_first else x
    want = x / torch.sqrt((x * x).mean(dim=2, keepdim=True) + 1e-5) * w.double() * (1 if gate_first else g)
    # half an ulp of bfloat16, and 32-bit arithmetic's 1e-6
    assert bool(((got.double().view(T, H, Dv) - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6 * float(want.abs().max())).all())
