"""The tiles of 128, 160 and 192 rows: edges of tiles, every epilogue, rotation, and the choice among tiles and pairs of launches."""
import pytest

from test_kernels_gpu import check_projection_with_rotation_and_cache_write, ops, rel      # noqa: F401  (ops is the fixture)

pytestmark = pytest.mark.gpu
TILES = {16: (128, 256), 27: (192, 192), 28: (192, 128), 29: (160, 256)}


@pytest.mark.parametrize("variant", sorted(TILES))
@pytest.mark.parametrize("dm,dn,K", [(0, 0, 192), (1, 4, 256), (-1, -4, 1024), (None, 20, 4160)])
def test_tiles_by_name(ops, variant, dm, dn, K):     # noqa: F811
    """One row and column more or less than whole tiles, and fewer rows than a tile; the fewest slices of K that the loop takes."""
    import torch
    from xyntetik_runner_amd.csrc.ops import KernelError
    bm, bn = TILES[variant]
    M, N = (5 if dm is None else 2 * bm + dm), 3 * bn + dn
    dev = torch.device("cuda:0")
    torch.manual_seed(variant * 10 + K)
    a = (torch.randn(M, K, device=dev) * 0.5).bfloat16()
    w = (torch.randn(N, K, device=dev) * 0.1).bfloat16()
    b = torch.randn(N, device=dev) * 0.1
    plain = a.double() @ w.double().T
    for wt in (w, ops.pack_weight(w)):
        got = ops.linear(a, wt, bias=b, out_dtype=torch.float32, variant=variant)
        assert rel(got, plain + b.double()) < 1e-5                                       # 32-bit sums
        for order in (1000, 2000):                                                       # the other orders of workgroups
            assert torch.equal(got, ops.linear(a, wt, bias=b, out_dtype=torch.float32, variant=order + variant))
        assert rel(ops.linear(a, wt, bias=b, variant=variant), plain + b.double()) < 6e-3     # rounded once to bfloat16
    base = torch.randn(M, N, device=dev)
    out = base.clone()
    ops.linear(a, w, out=out, accumulate=True, variant=variant)
    assert rel(out, base.double() + plain) < 1e-5
    w2 = (torch.randn(2 * N, K, device=dev) * 0.1).bfloat16()
    if variant == 27:       # an odd number of 32-column tiles a wave: gate and up do not meet
        with pytest.raises(KernelError, match="pair"):
            ops.linear_swiglu(a, w2, variant=variant)
    else:
        r = a.double() @ w2.double().T
        want = r[:, :N] / (1 + torch.exp(-r[:, :N])) * r[:, N:]
        for wt in (w2, ops.pack_weight(w2, gated=True)):
            assert rel(ops.linear_swiglu(a, wt, variant=variant), want) < 6e-3
    for bad in (72, 128):   # no whole slices, and fewer than three
        with pytest.raises(KernelError, match="four-wave"):
            ops.linear(a[:, :bad].contiguous(), w[:, :bad].contiguous(), variant=variant)


@pytest.mark.parametrize("variant", sorted(TILES))
@pytest.mark.parametrize("H,Hk,D,rot,inter", [(4, 2, 64, 64, False), (3, 1, 48, 32, False), (2, 1, 80, 80, True), (5, 1, 128, 128, False)])
def test_rotation_in_the_tiles_by_name(ops, variant, H, Hk, D, rot, inter):      # noqa: F811
    check_projection_with_rotation_and_cache_write(ops, "bfloat16", H, Hk, D, rot, inter, 16, [5, 0], [530, 70], True, 256, variant=variant)


@pytest.mark.parametrize("M", [137, 192, 193, 300, 321, 640, 1300, 1524])
@pytest.mark.parametrize("N,K", [(4096, 512), (12288, 256), (11008, 328), (22016, 512), (2048, 1376), (1024, 4096)])
def test_the_chosen_tiles(ops, M, N, K):      # noqa: F811
    """What the library chooses for sizes at which the new tiles, K ranges and two launches come in; K 328 is no whole slices, so
    that only the loops that look at columns take it, and nor is K 1376, which is split."""
    import torch
    dev = torch.device("cuda:0")
    torch.manual_seed(M + N + K)
    a = (torch.randn(M, K, device=dev) * 0.5).bfloat16()
    w = (torch.randn(N, K, device=dev) * 0.1).bfloat16()
    want = a.double() @ w.double().T
    assert rel(ops.linear(a, ops.pack_weight(w), out_dtype=torch.float32), want) < 1e-5
    half = N // 2 // 32 * 32
    gate, up = want[:, :half], want[:, half:2 * half]
    assert rel(ops.linear_swiglu(a, ops.pack_weight(w[:2 * half].contiguous(), gated=True)), gate / (1 + torch.exp(-gate)) * up) < 6e-3


@pytest.mark.parametrize("H,Hk,D,E,q_lens", [(12, 12, 64, 768, [600, 1448]), (16, 4, 128, 1000, [530, 70]), (8, 2, 80, 640, [513]), (40, 4, 128, 256, [1300])])
def test_rotation_in_the_chosen_tiles(ops, H, Hk, D, E, q_lens):      # noqa: F811
    check_projection_with_rotation_and_cache_write(ops, "bfloat16", H, Hk, D, D, False, 16, [0] * len(q_lens), q_lens, False, E)


# rows of one row of tiles (9 and 16 where tiles are wide products' way); column tiles enough for workgroups to begin at every slice of K and go round (K 256: as many slices as the
# loop has in flight), a K range each with streaming copies (17 rows) and without (64 rows)
@pytest.mark.parametrize("variant,M,N,K", [(0, 17, 5128, 256), (0, 64, 5128, 320), (58, 128, 5128, 256), (28, 192, 5128, 192), (55, 256, 5128, 192),
                                           (0, 9, 21504, 256), (0, 9, 32000, 4096), (0, 16, 21504, 4096), (0, 64, 20480, 4096), (0, 17, 2048, 8192), (0, 64, 2048, 8192), (0, 128, 21504, 1024)])
def test_one_row_of_tiles(ops, variant, M, N, K):      # noqa: F811
    import torch
    dev = torch.device("cuda:0")
    torch.manual_seed(M + N + K)
    a = (torch.randn(M, K, device=dev) * 0.5).bfloat16()
    w = (torch.randn(N, K, device=dev) * 0.1).bfloat16()
    want = a.double() @ w.double().T
    for wt in (w, ops.pack_weight(w)):
        assert rel(ops.linear(a, wt, out_dtype=torch.float32, variant=variant), want) < 1e-5
    half = N // 2 // 32 * 32
    w2 = w[:2 * half].contiguous()
    for wt in (w2, ops.pack_weight(w2, gated=True)):
        assert rel(ops.linear_swiglu(a, wt, variant=variant), want[:, :half] / (1 + torch.exp(-want[:, :half])) * want[:, half:2 * half]) < 6e-3
