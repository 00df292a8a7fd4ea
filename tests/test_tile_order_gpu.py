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


# 128 x 128 tiles: 9 and 16 row tiles (an eighth of the tiles an XCD), 17 (consecutive workgroups share a weight tile), fewer than 8 columns
@pytest.mark.parametrize("tiles_m,tiles_n", [(9, 11), (16, 8), (17, 9), (10, 3)])
@pytest.mark.parametrize("ragged", [0, 1])
def test_every_tile_of_many_rows_is_written(tiles_m, tiles_n, ragged):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(tiles_m * 100 + tiles_n + ragged)
    M, N, K = tiles_m * 128 - 37 * ragged, tiles_n * 128 - 20 * ragged, 256
    a, w = (torch.randn(s, generator=g, device=dev).bfloat16() for s in ((M, K), (N, K)))
    want = a.float() @ w.float().T
    bound = want.abs() * 2.0 ** -8 + K * 2.0 ** -24 * (a.float().abs() @ w.float().abs().T)
    for variant in (2017, 2117):
        out = torch.full((M, N), float("nan"), device=dev, dtype=torch.bfloat16)
        ops.linear(a, ops.pack_weight(w), out=out, variant=variant)
        assert ((out.float() - want).abs() <= bound).all(), f"variant {variant}"


# rows that are one row of tiles, two, some, and more than 16 of 128; columns of fewer tiles than XCDs, and no multiple of them
@pytest.mark.parametrize("M", [65, 129, 300, 520, 1100, 2100])
@pytest.mark.parametrize("N,K", [(200, 4096), (1000, 4160), (1536, 8192)])
def test_every_range_of_every_tile_is_added_once(M, N, K):
    """Few tiles and a long K: ranges of K beside each other, whatever their number.  (Room for the ranges' sums holds another
    product's sums, so that one left out would show.)"""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a, w = (torch.randn(s, generator=g, device=dev).bfloat16() for s in ((M, K), (2 * N, K)))
    ops.linear(a * 100, ops.pack_weight(w[:N].contiguous()))
    exact, size = a.float() @ w.float().T, a.float().abs() @ w.float().abs().T
    got = ops.linear(a, ops.pack_weight(w[:N].contiguous()), out_dtype=torch.float32)
    # 32-bit sums of exact products: 2^-24 of what has been added up, K times; and of the yardstick's as much
    assert ((got - exact[:, :N]).abs() <= 2 * K * 2.0 ** -24 * size[:, :N]).all()
    if N % 16 == 0:
        gate, up = exact[:, :N], exact[:, N:]
        both = ops.linear_swiglu(a, ops.pack_weight(w, gated=True) if N % 32 == 0 else w)
        want = torch.nn.functional.silu(gate) * up
        err = 2 * K * 2.0 ** -24 * (1.1 * size[:, :N] * up.abs() + gate.abs() * size[:, N:])       # (silu's slope is at most 1.1, and it at most its argument)
        assert ((both.float() - want).abs() <= err + want.abs() * 2.0 ** -8 + 1e-6).all()
