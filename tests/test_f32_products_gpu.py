"""The 32-bit product on the matrix cores and for few rows, at the edges of their tiles, runs and groups, against 64 bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows: one, the ends of the few-row kernel's groups, either side of its limit, of a tile's 32, 64 and 128; columns: less than a
# slice of 32, no multiple of it, either side of a run of 128; weight rows: few, no multiple of a tile, and so many that there are
# more than 256 tiles of 64 x 64 (one set of waves makes a tile then, two where there are fewer)
@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9, 16, 17, 33, 64, 65, 130, 200])
@pytest.mark.parametrize("N,K", [(7, 4), (96, 64), (100, 124), (65, 132), (200, 260), (16448, 68), (16450, 132)])
def test_product(M, N, K):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    rng = np.random.default_rng(M * 1000 + N + K)
    a, w, bias, c = rng.normal(size=(M, K + 8)), rng.normal(size=(N, K)), rng.normal(size=N), rng.normal(size=(M, N))
    t = lambda x: torch.tensor(x, dtype=torch.float32, device=dev)
    at = t(a)[:, 4:4 + K]                                  # rows that are part of wider ones
    exact = lambda x: x.double().cpu().numpy()
    want = exact(at) @ exact(t(w)).T
    # every product and sum rounds to 2^-24 of what has been added up so far: within K 2^-24 of the sum of magnitudes
    bound = (K + 4) * 2.0 ** -24 * (np.abs(exact(at)) @ np.abs(exact(t(w))).T + np.abs(bias) + np.abs(c))
    got = ops.linear(at, t(w))
    assert (np.abs(exact(got) - want) <= bound).all()
    with_bias = ops.linear(at, t(w), bias=t(bias))
    assert (np.abs(exact(with_bias) - (want + exact(t(bias)))) <= bound).all()
    out = t(c)
    ops.linear(at, t(w), out=out, accumulate=True)
    assert (np.abs(exact(out) - (want + exact(t(c)))) <= bound).all()
    # a row's result does not depend on the rows beside it, within a kernel's range of rows
    few = ops.linear(at[: max(1, M // 2)], t(w))
    if (M <= 16) == (few.shape[0] <= 16):
        assert torch.equal(few, got[: few.shape[0]])
    assert torch.equal(ops.linear(at, t(w), out_dtype=torch.bfloat16), got.bfloat16())


# the rows at which a few-row kernel ends, and weight rows and columns on either side of the lines between 2, 4 and 8 weight rows a wave
@pytest.mark.parametrize("M", [1, 3, 8, 16])
@pytest.mark.parametrize("N,K", [(4095, 256), (4097, 256), (6145, 260), (8191, 4096), (8193, 4096), (16383, 512), (16385, 512), (16385, 4096)])
def test_weight_rows_a_wave(M, N, K):
    """How many weight rows a wave takes changes no bit: the sums are those of narrow products, two weight rows a wave."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a, w = (torch.randn(s, generator=g, device=dev) for s in ((M, K), (N, K)))
    narrow = torch.cat([ops.linear(a, w[i:i + 2048]) for i in range(0, N, 2048)], dim=1)
    assert torch.equal(ops.linear(a, w), narrow)
    # and the sums themselves: K products and additions of 2^-24 each
    want, size = (a.double() @ w.double().T), (a.double().abs() @ w.double().abs().T)
    assert ((narrow.double() - want).abs() <= (K + 4) * 2.0 ** -24 * size).all()


# products that the library makes in tiles of two sets of waves and of four
@pytest.mark.parametrize("M,N,K", [(17, 1000, 4096), (17, 2048, 14336), (130, 1024, 8192), (401, 4096, 8192)])
def test_sums_of_one_sign_are_as_close_with_several_sets_of_waves(M, N, K):
    """Positive numbers, whose sums only grow: compensated sums of runs, however many sets of waves share the columns.  The tile that
    one set makes is the yardstick."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    assert ops.lib.xr_f32_tile(M, N, K) in (1, 2, 3)
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a, w = (torch.rand(s, generator=g, device=dev) for s in ((M, K), (N, K)))
    want = a.double() @ w.double().T
    off = lambda got: ((got.double() - want).norm() / want.norm()).item()
    one = off(ops.linear(a, w, variant=40))
    assert one < 2.0 ** -24                               # (what is left is the rounding inside a run)
    for tile in (1, 2, 3, 4):
        assert off(ops.linear(a, w, variant=40 + tile)) <= 1.02 * one         # (millions of roundings: their 2-norms agree to 1%)
    assert off(ops.linear(a, w)) <= 1.02 * one


# rows and weight rows at the edges of tiles, in the tiles that the library chooses for them: 32 x 32 with four sets, 32 x 64 and 64 x 64 with two;
# columns that are whole stages of one, two or four slices of 32, and that are not (516, 1028); fewer slices than a run (544)
@pytest.mark.parametrize("M,N", [(17, 31), (32, 2048), (33, 2050), (64, 4097), (401, 3072), (401, 2050), (300, 96), (130, 8200)])
@pytest.mark.parametrize("K", [516, 544, 1024, 1028, 2080])
def test_products_shared_by_sets_of_waves(M, N, K):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a, w, bias, c = (torch.randn(s, generator=g, device=dev) for s in ((M, K + 4), (N, K), (N,), (M, N)))
    a = a[:, 4:]
    want = a.double() @ w.double().T
    # (each product and sum rounds to 2^-24 of what has been added up so far)
    bound = (K + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs() + c.double().abs())
    assert ((ops.linear(a, w).double() - want).abs() <= bound).all()
    assert ((ops.linear(a, w, bias=bias).double() - want - bias.double()).abs() <= bound).all()
    out = c.clone()
    ops.linear(a, w, out=out, accumulate=True)
    assert ((out.double() - want - c.double()).abs() <= bound).all()
    a[0, K // 2] = float("inf")
    got = ops.linear(a, w)
    assert not torch.isfinite(got[0]).any() and not torch.isnan(got[0][w[:, K // 2] != 0]).any()      # (an infinite sum stays infinite)
    assert ((got[1:].double() - want[1:]).abs() <= bound[1:]).all()


# every tile by number (xr_f32_tile's: 32 x 128 with one set of waves, 64 x 64 and 32 x 64 with two, 32 x 32 with four, 64 x 64 in runs of 64
# columns): rows and weight rows short of a tile, one past it and many; K that is whole stages of one, two and four slices, and that is not
@pytest.mark.parametrize("tile", range(5))
@pytest.mark.parametrize("M,N,K", [(17, 31, 516), (33, 129, 1024), (65, 2050, 2080), (130, 515, 1028), (401, 2050, 768), (64, 28675, 544)])
def test_tiles_by_number(tile, M, N, K):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a, w, bias, c = (torch.randn(s, generator=g, device=dev) for s in ((M, K + 4), (N, K), (N,), (M, N)))
    a = a[:, 4:]
    want = a.double() @ w.double().T
    # (each product and sum rounds to 2^-24 of what has been added up so far)
    bound = (K + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs() + c.double().abs())
    got = ops.linear(a, w, variant=40 + tile)
    assert ((got.double() - want).abs() <= bound).all()
    # a run of at most 128 columns is one sum, the runs' sums are compensated: a root mean square error of less than 4 units of 2^-24 of it
    assert ((got.double() - want).norm() / want.norm()).item() < 4 * 2.0 ** -24
    assert torch.equal(ops.linear(a, w, out_dtype=torch.bfloat16, variant=40 + tile), got.bfloat16())
    assert ((ops.linear(a, w, bias=bias, variant=40 + tile).double() - want - bias.double()).abs() <= bound).all()
    out = c.clone()
    ops.linear(a, w, out=out, accumulate=True, variant=40 + tile)
    assert ((out.double() - want - c.double()).abs() <= bound).all()
    a[0, K // 2] = float("inf")
    got = ops.linear(a, w, variant=40 + tile)
    assert not torch.isfinite(got[0]).any() and not torch.isnan(got[0][w[:, K // 2] != 0]).any()      # (an infinite sum stays infinite)
    assert ((got[1:].double() - want[1:]).abs() <= bound[1:]).all()


# no branch of the choice is left without a product: wide heads of few rows, few runs of columns in many and in few tiles, and the four lines
# between 512 and 1,024 columns
@pytest.mark.parametrize("M,N,K,tile", [(17, 128256, 2048, 0), (1024, 8192, 260, 0), (401, 16384, 2048, 1), (401, 128256, 2048, 0), (300, 2048, 516, 4),
                                        (33, 12288, 1024, 1), (401, 3072, 2048, 2), (64, 2048, 8192, 3), (20, 64, 64, 2), (64, 768, 768, 3), (401, 768, 768, 3), (401, 900, 768, 2),
                                        (1024, 768, 768, 4), (128, 6144, 768, 4), (401, 2304, 768, 1)])
def test_the_chosen_tile(M, N, K, tile):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    assert ops.lib.xr_f32_tile(M, N, K) == tile
    a, w = torch.randn(M, K, device=dev), torch.randn(N, K, device=dev)
    assert torch.equal(ops.linear(a, w), ops.linear(a, w, variant=40 + tile))
