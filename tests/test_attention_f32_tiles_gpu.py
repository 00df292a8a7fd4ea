"""32-bit attention at the edges of its tiles of 64 keys, of 32 rows and of the pieces that a thread moves, against 64 bits."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_kernels_gpu import DEV, FakeCtx, fill_cache, scatter_pages


# head and value sizes: one piece a thread, whole and not; four, whole and not; eight; values wider and narrower than keys
@pytest.mark.parametrize("H,Hk,D,Dv", [(2, 2, 4, 12), (4, 2, 16, 16), (6, 2, 20, 64), (4, 1, 64, 64), (8, 2, 64, 20), (3, 3, 68, 48), (2, 1, 128, 128), (2, 1, 12, 120)])
@pytest.mark.parametrize("mask", [{}, {"window": 70}, {"chunk": 100}, {"window": 40, "keep_first": 66}, {"window": 3, "keep_first": 130}])
@pytest.mark.parametrize("ps", [4, 64])
def test_tiles(H, Hk, D, Dv, mask, ps):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    g = torch.Generator()
    g.manual_seed(H + D + Dv + ps)
    starts, q_lens = [0, 63, 150, 0], [70, 2, 65, 1]            # first tiles, one past a tile, several, a lone token
    lens = [s + n for s, n in zip(starts, q_lens)]
    tables, n_pages = scatter_pages(lens, ps, 2)
    ctx = FakeCtx(starts, q_lens, tables, ps)
    q = torch.randn(sum(q_lens), H * D, generator=g)
    ks, vs = [torch.randn(n, Hk, D, generator=g) for n in lens], [torch.randn(n, Hk, Dv, generator=g) for n in lens]
    kc, vc = fill_cache(ks, ks, tables, n_pages, ps, torch.float32)[0], fill_cache(vs, vs, tables, n_pages, ps, torch.float32)[1]
    got = ops.attention(q.to(DEV), kc, vc, ctx, 0, H, Hk, D, ps, 1 / math.sqrt(D), v_head_dim=Dv, **mask).cpu().double().numpy().reshape(-1, H, Dv)
    t = 0
    for k, v, s, n in zip(ks, vs, starts, q_lens):
        k, v = k.double().numpy(), v.double().numpy()
        for p in range(s, s + n):
            lo = p - p % mask["chunk"] if "chunk" in mask else max(0, p - mask.get("window", p + 1) + 1)
            seen = [j for j in range(p + 1) if j >= lo or j < mask.get("keep_first", 0)]
            for h in range(H):
                x = k[seen, h // (H // Hk)] @ q[t].double().numpy().reshape(H, D)[h] / math.sqrt(D)
                w = np.exp(x - x.max())
                w /= w.sum()
                # a score rounds D products and sums to 2^-24 of at most sum |q k| / sqrt(D) < 16, as its exponential's factor; the weighted
                # sum rounds once a key
                bound = (16 * (D + 4) + len(seen) + 8) * 2.0 ** -24 * (w @ np.abs(v[seen, h // (H // Hk)])) + 1e-30
                assert (np.abs(got[t, h] - w @ v[seen, h // (H // Hk)]) <= bound).all(), (p, h)
            t += 1


@pytest.mark.parametrize("H,Hk,D", [(2, 2, 16), (2, 2, 32), (8, 2, 64)])
def test_rows_beside_a_row(H, Hk, D):
    """Four rows of a workgroup and fewer take their softmax with a wave each, more with eight lanes each: the same bits."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    g = torch.Generator()
    g.manual_seed(D)
    n, ps = 200, 16
    tables, n_pages = scatter_pages([n], ps, 2)
    q, k, v = torch.randn(n, H * D, generator=g), torch.randn(n, Hk, D, generator=g), torch.randn(n, Hk, D, generator=g)
    kc, vc = fill_cache([k], [k], tables, n_pages, ps, torch.float32)[0], fill_cache([v], [v], tables, n_pages, ps, torch.float32)[1]
    run = lambda a, b: ops.attention(q[a:b].to(DEV), kc, vc, FakeCtx([a], [b - a], tables, ps), 0, H, Hk, D, ps, 1 / math.sqrt(D))
    whole = run(0, n)
    for a, b in ((0, 1), (63, 64), (64, 66), (120, 124), (128, 133), (199, 200)):
        assert torch.equal(run(a, b), whole[a:b]), (a, b)
