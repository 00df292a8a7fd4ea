"""The kernels that add a product's K ranges up and norm, or rotate and cache, the result: rows on either side of what a thread keeps in
registers, and rotations with and without a step's table."""
import pytest

pytestmark = pytest.mark.gpu

from test_kernels_gpu import DEV, FakeCtx, scatter_pages


# rows of one group of four columns a thread, its last missing, two, and longer
@pytest.mark.parametrize("N", [68, 4096, 4100, 8192, 8196])
@pytest.mark.parametrize("M", [17, 130])
@pytest.mark.parametrize("centred", [False, True])
def test_norm(M, N, centred):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    g = torch.Generator(device=DEV)
    g.manual_seed(M + N)
    K = 512
    a, w, x, nw, b = (torch.randn(s, generator=g, device=DEV) for s in ((M, K), (N, K), (M, N), (N,), (N,)))
    a, w = a.bfloat16(), (w * 0.05).bfloat16()
    x = x * torch.linspace(0.1, 30, M, device=DEV)[:, None] + 1
    want = x.double() + a.double() @ w.double().T + b.double()
    size = x.double().abs() + a.double().abs() @ w.double().abs().T + b.double().abs()
    got = x.clone()
    h = ops.linear_add_rmsnorm(a, ops.pack_weight(w), got, nw, 1e-5, torch.bfloat16, bias=b, centred=centred)
    assert ((got.double() - want).abs() <= (K + 8) * 2.0 ** -24 * size).all()
    y = got.double() - (got.double().mean(1, keepdim=True) if centred else 0)
    norm = y * torch.rsqrt((y * y).mean(1, keepdim=True) + 1e-5) * nw.double()
    # (bfloat16 rounds to 2^-9; a mean of N numbers up to N 2^-24 of them off)
    assert ((h.double() - norm).abs() <= 2.0 ** -8 * norm.abs() + 2.0 ** -14 * nw.double().abs()).all()
    # the post-norm's rows: the same kernel, whose rows are the normed ones
    if not centred:
        z, out = x.clone(), x.double() * 0.5 + a.double() @ w.double().T
        h = ops.linear_post_norm(a, ops.pack_weight(w), z, 0.5, nw, 1e-5, torch.bfloat16)
        out = out * torch.rsqrt((out * out).mean(1, keepdim=True) + 1e-5) * nw.double()
        assert ((z.double() - out).abs() <= 2.0 ** -14 * (out.abs() + nw.double().abs())).all() and torch.equal(h, z.bfloat16())


@pytest.mark.parametrize("T", [17, 70, 200])
@pytest.mark.parametrize("H,Hk,D,rot,inter,ps", [(4, 2, 64, 64, False, 64), (4, 4, 48, 32, False, 16), (2, 1, 128, 128, True, 32), (3, 1, 16, 6, True, 4), (2, 0, 64, 64, False, 16),
                                                 (4, 2, 32, 0, False, 16)])
def test_rotation(T, H, Hk, D, rot, inter, ps):
    """With the step's table and without it the same bits, and the product and the rotation's own kernel one after the other."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    g = torch.Generator(device=DEV)
    g.manual_seed(T + D + rot)
    starts, q_lens = [5, 0, 131], [T - 9, 1, 8]
    tables, n_pages = scatter_pages([s + n for s, n in zip(starts, q_lens)], ps, 2)
    ctx = FakeCtx(starts, q_lens, tables, ps)
    Q, K = H * D, Hk * D
    h = torch.randn(T, 256, generator=g, device=DEV).bfloat16()
    w = ops.pack_weight((torch.randn(Q + 2 * K, 256, generator=g, device=DEV) * 0.1).bfloat16())
    b = torch.randn(Q + 2 * K, generator=g, device=DEV)
    inv = (10000.0 ** (-torch.arange(rot // 2, dtype=torch.float64) * 2 / rot)).float().to(DEV) if rot else None
    paired = rot > 0 and not inter
    results, asked = [], []

    def table():
        asked.append(1)
        return ops.rope_table(ctx.positions, inv, 1.0)
    for how in ("table", "none", "apart"):
        kc, vc = (torch.full((n_pages, max(Hk, 1)) + s, 7.0, device=DEV, dtype=torch.bfloat16) for s in ((ps, D), (D, ps)))
        ops.fuse_rope = how != "apart"
        try:
            q = ops.project_rope_kv_write(h, w, b, kc if Hk else None, vc if Hk else None, ctx.positions, ctx.req_of_token, ctx.block_table(0), inv,
                                          H, Hk, D, rot, inter, 1.0, ps, paired=paired, finish_table=table if how == "table" and rot else None)
        finally:
            ops.fuse_rope = True
        results.append((q, kc, vc))
    assert len(asked) == (1 if rot else 0)
    for one, two, three in zip(*results):
        assert torch.equal(one, two)
        # (the product's sums in another order, both rounded to bfloat16)
        assert ((one.double() - three.double()).abs() <= 2.0 ** -7 * three.double().abs() + 2.0 ** -9).all()


@pytest.mark.parametrize("T", [17, 130, 511])
@pytest.mark.parametrize("H,Hk,D,rot,inter", [(4, 2, 64, 64, False), (2, 1, 48, 32, False), (3, 1, 16, 6, True)])
def test_keys_that_are_not_8_byte_aligned(T, H, Hk, D, rot, inter):
    """The kernel that stores four channels at a time does not take them; one column a thread does, with the same sums."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, ps = load_ops(), 16
    g = torch.Generator(device=DEV)
    g.manual_seed(T + D)
    tables, n_pages = scatter_pages([T + 3], ps, 2)
    ctx = FakeCtx([3], [T], tables, ps)
    h = torch.randn(T, 256, generator=g, device=DEV).bfloat16()
    w = ops.pack_weight((torch.randn((H + 2 * Hk) * D, 256, generator=g, device=DEV) * 0.1).bfloat16())
    inv = (10000.0 ** (-torch.arange(rot // 2, dtype=torch.float64) * 2 / rot)).float().to(DEV)
    results = []
    for shift in (0, 1):
        size = n_pages * Hk * ps * D
        kc = torch.full((size + 8,), 7.0, device=DEV, dtype=torch.bfloat16)[shift:shift + size].view(n_pages, Hk, ps, D)
        vc = torch.full((n_pages, Hk, D, ps), 7.0, device=DEV, dtype=torch.bfloat16)
        assert kc.data_ptr() % 8 == 2 * shift
        q = ops.project_rope_kv_write(h, w, None, kc, vc, ctx.positions, ctx.req_of_token, ctx.block_table(0), inv, H, Hk, D, rot, inter, 1.0, ps,
                                      paired=not inter, finish_table=lambda: ops.rope_table(ctx.positions, inv, 1.0))
        results.append((q, kc, vc))
    assert torch.equal(results[0][2], results[1][2])
    for one, two in zip(*results):
        # (a rotation's two products and their sum, in 32 bits in another order, then a bfloat16 rounding)
        assert ((one.double() - two.double()).abs() <= 2.0 ** -8 * two.double().abs() + 2.0 ** -18).all()
