"""The order of a product's tiles over the XCDs: every tile is made once, whether the shares are whole columns or not."""
import pytest

pytestmark = pytest.mark.gpu


# rows and columns of 256 x 256 tiles: 6 x 42 and 3 x 85 (whole columns would give an XCD a round more than an even share), 5 x 51
# (the shares are not equal), 7 x 9 and 8 x 8 (whole columns), each with a ragged last tile too
@pytest.mark.parametrize("tiles_m,tiles_n", [(6, 42), (3, 85), (5, 51), (7, 9), (8, 8)])
@pytest.mark.parametrize("ragged", [0, 1])
def test_every_tile_is_written(tiles_m, tiles_n, ragged):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(tiles_m * 100 + tiles_n + ragged)
    M, N, K = tiles_m * 256 - 37 * ragged, tiles_n * 256 - 20 * ragged, 128
    a = torch.randn((M, K), generator=g, device=dev).bfloat16()
    w = torch.randn((N, K), generator=g, device=dev).bfloat16()
    want = a.float() @ w.float().T
    # 32-bit sums of exact products, rounded once to bfloat16: half a unit in the last place, and the order of 128 sums
    bound = want.abs() * 2.0 ** -8 + K * 2.0 ** -24 * (a.float().abs() @ w.float().abs().T)
    for variant in (2014, 2114, 0):
        out = torch.full((M, N), float("nan"), device=dev, dtype=torch.bfloat16)
        ops.linear(a, ops.pack_weight(w), out=out, variant=variant)
        assert ((out.float() - want).abs() <= bound).all(), f"variant {variant}"
