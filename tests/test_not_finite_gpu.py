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
