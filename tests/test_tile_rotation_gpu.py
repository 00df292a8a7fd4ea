"""Tiles that rotate what they write: cosines and sines in LDS for all rows, for 32 rows of each wave, or from memory; values whose
aligned groups of positions begin at any row."""
import pytest

from test_kernels_gpu import check_projection_with_rotation_and_cache_write, ops      # noqa: F401  (ops is the fixture)

pytestmark = pytest.mark.gpu


# 12, 14, 26: eight waves, four of them along rows (a table of 32 rows of each: up to 128 x 1 KB do not fit); 17, 27: four waves (all
# rows' table of 128 channels fits, of 256 a part); 29: one wave along rows.  Odd numbers of pairs, whose table is copied
# pair by pair, and heads that are rotated in part of 16 columns.
@pytest.mark.parametrize("variant", [12, 14, 17, 26, 27, 29])
@pytest.mark.parametrize("H,Hk,D,rot,inter,ps", [(3, 1, 128, 128, False, 16), (2, 1, 256, 256, False, 8), (1, 1, 256, 254, True, 16), (3, 2, 48, 18, True, 4),
                                                 (2, 1, 64, 6, True, 16), (2, 2, 96, 16, False, 32), (2, 1, 64, 0, False, 16)])
def test_tables_and_row_groups(ops, variant, H, Hk, D, rot, inter, ps):      # noqa: F811
    check_projection_with_rotation_and_cache_write(ops, "bfloat16", H, Hk, D, rot, inter, ps, [3, 0, 7], [257, 11, 250], D == 96, 256, variant=variant)


def test_keys_that_are_not_16_byte_aligned(ops):      # noqa: F811
    """Tiles store 8 channels at a time; a cache that begins 8 bytes later takes the product and the rotation's own kernel."""
    import torch
    from test_kernels_gpu import DEV, FakeCtx, scatter_pages
    torch.manual_seed(5)
    H, Hk, D, ps, T = 2, 1, 64, 16, 520
    tables, n_pages = scatter_pages([T], ps, 2)
    ctx = FakeCtx([0], [T], tables, ps)
    h = torch.randn(T, 256, device=DEV).bfloat16()
    w = ops.pack_weight((torch.randn((H + 2 * Hk) * D, 256, device=DEV) * 0.1).bfloat16())
    inv = (10000.0 ** (-torch.arange(D // 2, dtype=torch.float64) * 2 / D)).float().to(DEV)
    results = []
    for shift, fuse in ((0, False), (4, True)):
        size = n_pages * Hk * ps * D
        kc = torch.full((size + 8,), 7.0, device=DEV, dtype=torch.bfloat16)[shift:shift + size].view(n_pages, Hk, ps, D)
        vc = torch.full((n_pages, Hk, D, ps), 7.0, device=DEV, dtype=torch.bfloat16)
        assert kc.data_ptr() % 16 == 2 * shift
        ops.fuse_rope = fuse
        try:
            q = ops.project_rope_kv_write(h, w, None, kc, vc, ctx.positions, ctx.req_of_token, ctx.block_table(0), inv, H, Hk, D, D, False, 1.0, ps,
                                          paired=True)
        finally:
            ops.fuse_rope = True
        results.append((q, kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_pages_of_more_than_32_bits_channels(ops):      # noqa: F811
    """A page of 2^20 positions of 16 heads of 256: 2^32 channels."""
    import torch
    from test_kernels_gpu import DEV, FakeCtx
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("two pages of keys and of values are 32 GiB")
    torch.manual_seed(6)
    H, Hk, D, ps, T = 1, 16, 256, 1 << 20, 520
    ctx = FakeCtx([3], [T], [[1]], ps)
    h = torch.randn(T, 256, device=DEV).bfloat16()
    w = ops.pack_weight((torch.randn((H + 2 * Hk) * D, 256, device=DEV) * 0.1).bfloat16())
    inv = (10000.0 ** (-torch.arange(D // 2, dtype=torch.float64) * 2 / D)).float().to(DEV)
    kc, vc = (torch.empty((2, Hk) + s, device=DEV, dtype=torch.bfloat16) for s in ((ps, D), (D, ps)))
    results = []
    for fuse in (False, True):
        kc[:, :, :3 + T], vc[..., :3 + T] = 7.0, 7.0
        ops.fuse_rope = fuse
        try:
            q = ops.project_rope_kv_write(h, w, None, kc, vc, ctx.positions, ctx.req_of_token, ctx.block_table(0), inv, H, Hk, D, D, False, 1.0, ps,
                                          paired=True)
        finally:
            ops.fuse_rope = True
        results.append([x.clone() for x in (q, kc[:, :, :3 + T], vc[..., :3 + T])])
    for one, two in zip(*results):
        # (the same product in tiles, both rounded to bfloat16)
        assert ((one.double() - two.double()).abs() <= 2.0 ** -7 * one.double().abs() + 2.0 ** -9).all()
