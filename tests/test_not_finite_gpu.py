"""Values that are no finite numbers show where they belong and nowhere else: the true 32-bit path is there to show faults, and a
fault must not move to another token on its way."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_kernels_gpu import DEV, FakeCtx, fill_cache, scatter_pages


def same(got, want, tol, what=""):
    """Finite values close, all others alike (NaN, infinite of either sign), place by place."""
    got, want = np.asarray(got, dtype=np.float64), np.asarray(want, dtype=np.float64)
    ok = np.isfinite(want)
    assert (np.isnan(got) == np.isnan(want)).all() and (np.isposinf(got) == np.isposinf(want)).all(), f"{what}: not finite elsewhere"
    assert (np.isneginf(got) == np.isneginf(want)).all(), f"{what}: infinite elsewhere"
    assert np.abs(got[ok] - want[ok]).max() <= tol * np.abs(want[ok]).max(), what


@pytest.mark.parametrize("H,Hk,D,Dv", [(4, 2, 32, 32), (3, 3, 16, 128), (8, 1, 128, 48)])
@pytest.mark.parametrize("mask", [{}, {"window": 24}, {"chunk": 40}, {"window": 24, "keep_first": 3}])
def test_attention_in_32_bits(H, Hk, D, Dv, mask):
    """Tokens before one whose value is not finite do not see it, nor do those whose window or chunk has passed it."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    torch.manual_seed(D + Dv)
    starts, q_lens, ps = [5, 0, 70], [90, 40, 1], 16
    lens = [s + n for s, n in zip(starts, q_lens)]
    tables, n_pages = scatter_pages(lens, ps, 2)
    ctx = FakeCtx(starts, q_lens, tables, ps)
    q = torch.randn(sum(q_lens), H * D)
    k_seq, v_seq = [torch.randn(n, Hk, D) for n in lens], [torch.randn(n, Hk, Dv) for n in lens]
    v_seq[0][60, 0, 3], v_seq[0][61, Hk - 1, 5], v_seq[0][80, Hk - 1, 7] = math.inf, math.nan, -math.inf
    v_seq[1][20, 0, 15], v_seq[1][1, Hk - 1, 0], v_seq[2][30, 0, 1] = math.nan, math.inf, -math.inf
    kc, vc = fill_cache(k_seq, k_seq, tables, n_pages, ps, torch.float32)[0], fill_cache(v_seq, v_seq, tables, n_pages, ps, torch.float32)[1]
    got = ops.attention(q.to(DEV), kc, vc, ctx, 0, H, Hk, D, ps, 1 / math.sqrt(D), v_head_dim=Dv, **mask)
    want, t = np.zeros((sum(q_lens), H, Dv)), 0
    for b, (s, n) in enumerate(zip(starts, q_lens)):
        k, v = k_seq[b].double().numpy(), v_seq[b].double().numpy()
        for p in range(s, s + n):
            lo = p - p % mask["chunk"] if "chunk" in mask else max(0, p - mask.get("window", p + 1) + 1)
            seen = [j for j in range(p + 1) if j >= lo or j < mask.get("keep_first", 0)]
            for h in range(H):
                kv = h // (H // Hk)
                x = k[seen, kv] @ q[t].double().numpy().reshape(H, D)[h] / math.sqrt(D)
                w = np.exp(x - x.max())
                with np.errstate(invalid="ignore"):
                    want[t, h] = (w[:, None] / w.sum() * v[seen, kv]).sum(0)
            t += 1
    # 32-bit sums over up to 95 keys of weights that sum to one: a few 2^-24 times sqrt(95), scores within 1e-5 of theirs
    same(got.cpu().numpy().reshape(want.shape), want, 2e-5, str(mask))


@pytest.mark.parametrize("kind,where", [(k, w) for k in ("delta", "retention") for w in ("q", "k", "v", "decay", "negative decay", "big")]
                         + [("delta", "beta")])
@pytest.mark.parametrize("D,Dv", [(48, 16), (128, 32)])
def test_recurrences_in_chunks(monkeypatch, kind, where, D, Dv):
    """Rows before one with an infinity or a NaN, in the middle of a chunk, are as they are without it; the rows behind it and the
    state are what the recurrence makes of it token by token.  A negative decay is one like another."""
    from xyntetik_runner_amd.csrc.ops import load_ops
    from test_recurrence_chunks_gpu import PORTIONS, both
    ops = load_ops()
    H = 2
    rng = np.random.default_rng(D)
    lens = [sum(n for _, n in p) for p in PORTIONS]
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    unit = lambda x: x / np.linalg.norm(x, axis=-1, keepdims=True)
    qs, ks = ([f32(unit(rng.normal(size=(n, H, D)))) for n in lens] for _ in range(2))
    vs = [f32(rng.normal(size=(n, H, Dv))) for n in lens]
    beta, gate = ([f32(x + 0.5 * rng.uniform(size=(n, H))) for n in lens] for x in (0.25, 0.5))
    decay = f32(np.array([0.97, 0.9]))
    bad = {"q": qs, "k": ks, "v": vs, "beta": beta}.get(where)
    if bad is not None:
        bad[0][137].flat[1], bad[0][299].flat[0], bad[1][20].flat[-1] = np.inf, np.nan, -np.inf
        bad[2][127].flat[0], bad[3][0].flat[0] = np.nan, np.inf
    elif where == "decay":
        gate[0][137, 1] = gate[2][128, 0] = decay[1] = np.nan
    elif where == "negative decay":
        gate[0][[137, 138, 190], 1], gate[1][64, 0], decay[1] = -0.5, -1.0, -0.9
    else:                               # sums that pass the largest number on the way
        vs[0][130:140, 1, 2], ks[0][130:140, 1] = 3e38, ks[0][130, 1]
    extra = (beta, gate) if kind == "delta" else decay
    chunks, plain = both(ops, monkeypatch, kind, qs, ks, vs, extra, H, H, D, Dv, PORTIONS, [2, 0, 4, 1], 5)
    for b, (got, want) in enumerate(zip(chunks, plain)):
        if where != "big":
            same(got, want, 2e-5, f"request {b}")
        else:                           # (where a sum overflows depends on its order: the rows before, and the other columns)
            same(got[:130], want[:130], 2e-5, f"request {b}")
            same(np.delete(got, 2, axis=2), np.delete(want, 2, axis=2), 2e-5, f"request {b}")


# rows for the few-row kernel, for tiles of two sets of waves, of one, and 64 x 128 of them; a row stride that is no multiple of four
# (the kernel without matrix cores); one run of columns, several, and a rest
@pytest.mark.parametrize("M,N,aligned", [(5, 96, True), (17, 100, True), (130, 16448, True), (260, 16448, True), (40, 100, False)])
@pytest.mark.parametrize("K", [64, 128, 200, 384])
def test_products_in_32_bits(M, N, aligned, K):
    """A product or a sum past the largest number is infinite, whichever columns it comes from, a NaN stays one, and no other
    row or column is touched."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(K + M)
    a, w = (rng.normal(size=s).astype(np.float32) for s in ((M, K), (N, K)))
    a[1, 3], w[:, 3] = 3e38, 2.0 + np.abs(w[:, 3])                       # a product, in the first run
    a[2, K - 1], w[:, K - 1] = -3e38, 2.0 + np.abs(w[:, K - 1])          # and the last column, to the other side
    a[3, [5, 40]], w[:, [5, 40]] = 2e38, 1.0                             # a sum of two, from the two sets' slices of 32
    a[4, K // 2] = np.nan
    w[7, K // 2 + 1] = np.inf
    row = torch.zeros((M, K + (8 if aligned else 5)), device=DEV)
    row[:, 4:4 + K] = torch.tensor(a)
    got = ops.linear(row[:, 4:4 + K], torch.tensor(w, device=DEV)).cpu().numpy()
    with np.errstate(over="ignore", invalid="ignore"):
        want = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32)
    same(np.delete(got, [1, 2, 3], axis=0), np.delete(want, [1, 2, 3], axis=0), 2e-5)
    for r, sign in ((1, 1), (2, -1), (3, 1)):
        assert (np.delete(got[r], 7) == sign * np.inf).all(), f"row {r}"
