"""32-bit products made of bfloat16 parts on the matrix cores, at the edges of their tiles and ranges of K, against 64 bits and the 32-bit kernel."""
import pytest

pytestmark = pytest.mark.gpu

TILES, U = 4, 2.0 ** -24


def plan(tile, ranges):
    return 60 + 1 + tile + TILES * (ranges - 1)


def operands(M, N, K, kind="normal"):
    import torch
    from xyntetik_runner_amd.csrc.ops import F32Weight, load_ops
    g = torch.Generator(device="cuda:0")
    g.manual_seed(M + N + K)
    make = torch.rand if kind == "one sign" else torch.randn
    a, w, bias, c = (make(s, generator=g, device="cuda:0") for s in ((M, K + 4), (N, K), (N,), (M, N + 3)))
    if kind == "wide":
        a = a * torch.exp(3 * torch.randn(a.shape, generator=g, device="cuda:0"))
    return load_ops(), a[:, 4:], w.as_subclass(F32Weight), bias, c[:, 3:]              # (rows that are part of wider ones)


# rows and weight rows: one past the few-row kernels, short of a tile, whole tiles, one past; K: one pair of slabs, a run, one past it, several;
# ranges: none, even ones, a last one that is shorter
@pytest.mark.parametrize("M,N,K", [(17, 1, 64), (32, 128, 256), (33, 129, 320), (65, 70, 512), (128, 128, 1088), (130, 515, 2048), (257, 200, 640)])
def test_tiles_and_ranges(M, N, K):
    import torch
    ops, a, w, bias, c = operands(M, N, K)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    # a run is 16 additions of 2^-24 of what has been added up so far (twice that, for what an instruction may round inside), the runs' sums lose
    # a few 2^-24 more, the products left out at most 2^-24 (of ordinary numbers together about 2^-26)
    bound = 40 * U * size
    whole = None
    for tile in range(TILES):
        for ranges in (1, 2, 3, 5):
            if ranges > K // 64:
                continue
            v = plan(tile, ranges)
            got = ops.linear(a, w, variant=v)
            assert ((got.double() - want).abs() <= bound).all()
            if ranges == 1:                                     # a result does not depend on the tile, nor on the rows beside it
                whole = got if whole is None else whole
                assert torch.equal(got, whole)
                assert torch.equal(ops.linear(a[:17], w, variant=v), whole[:17])
            assert torch.equal(ops.linear(a, w, out_dtype=torch.bfloat16, variant=v), got.bfloat16())
            assert torch.equal(ops.linear(a, w, bias=bias, variant=v), got + bias)
            out = c.clone()
            ops.linear(a, w, out=out, accumulate=True, variant=v)
            assert torch.equal(out, got + c)
            wide = torch.empty_like(c.repeat(1, 2))[:, 1:1 + N]
            assert torch.equal(ops.linear(a, w, out=wide, variant=v), got)


# as the library chooses: no further from 64 bits than the 32-bit instructions' kernel, whatever the numbers' signs and sizes
@pytest.mark.parametrize("kind", ["normal", "one sign", "wide"])
@pytest.mark.parametrize("M,N,K", [(17, 2048, 8192), (100, 16384, 2048), (401, 4096, 8192), (700, 3072, 768)])
def test_no_further_from_the_exact_product(M, N, K, kind):
    ops, a, w, _, _ = operands(M, N, K, kind)
    assert ops.lib.xr_gemm_f32_parts_plan(M, N, K) > 0
    want = a.double() @ w.double().T
    off = lambda got: ((got.double() - want).norm() / want.norm()).item()
    assert off(ops.linear(a, w)) <= min(off(ops.linear(a, w, variant=40 + t)) for t in range(4))


@pytest.mark.parametrize("ranges", [1, 3])
@pytest.mark.parametrize("tile", range(TILES))
def test_numbers_at_the_ends_of_the_range(tile, ranges):
    """Infinities, NaNs, sums that overflow, numbers beside bfloat16's largest, and numbers whose parts are too small for bfloat16: the
    32-bit kernel's results."""
    import torch
    M, N, K = 140, 150, 576
    ops, a, w, _, _ = operands(M, N, K)
    a = a.clone()
    a[0, 5], a[3, 70], a[70, 300], a[139, K - 1] = float("inf"), float("nan"), float("-inf"), 3.4e38
    a[5, 0], a[5, 40] = 3e38, 3e38
    w[:, 0], w[:, 40], w[:, K - 1] = 1.0, 1.0, 0.5              # (in place: the weight's own memory)
    w[7, 5] = 0.0                                               # infinity times zero
    a[20:22] *= 1e-36
    w[100:102] *= 1e-33
    got, want = (ops.linear(a, w, variant=v) for v in (plan(tile, ranges), 40))
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])
    fin = torch.isfinite(want)
    size = (a.double().abs() @ w.double().abs().T).clamp(max=1e38)
    assert ((got.double() - want.double()).abs()[fin] <= (80 * U * size + K * 2.0 ** -149)[fin]).all()     # (a product below 2^-126 rounds to 2^-149)


@pytest.mark.parametrize("ranges", [1, 3])
@pytest.mark.parametrize("tile", range(TILES))
def test_a_result_depends_on_its_own_row_and_column(tile, ranges):
    """What is no ordinary number in some rows and weight rows (an infinity, a NaN, an overflow, tiny numbers, zeros) changes no bit elsewhere."""
    import torch
    M, N, K = 140, 150, 576
    ops, a, w, _, _ = operands(M, N, K)
    want = ops.linear(a, w, variant=plan(tile, ranges))
    odd, odd_w = a.clone(), w.as_subclass(torch.Tensor).clone()
    odd[0, 5], odd[37, 70], odd[70, 300], odd[139, K - 1] = float("inf"), float("nan"), 3.4e38, float("-inf")
    odd[64] *= 1e-30
    odd[100] = 0.0
    odd_w[3, 9], odd_w[149, 0] = float("inf"), float("nan")
    odd_w[90] *= 1e-30
    got = ops.linear(odd, odd_w.as_subclass(type(w)), variant=plan(tile, ranges))
    rows = [m for m in range(M) if m not in (0, 37, 64, 70, 100, 139)]
    cols = [n for n in range(N) if n not in (3, 90, 149)]
    assert torch.equal(got[rows][:, cols], want[rows][:, cols])


@pytest.mark.parametrize("ranges", [1, 3])
@pytest.mark.parametrize("tile", range(TILES))
def test_tiny_numbers_that_meet_large_ones(tile, ranges):
    """Numbers whose parts are below bfloat16's range count where the others are large: every bit of them, as with 32-bit products."""
    import torch
    M, N, K = 140, 150, 576
    ops, a, w, _, _ = operands(M, N, K)
    a, w = a.clone(), w.as_subclass(torch.Tensor).clone()
    a[20:23] *= torch.tensor([1e-36, 1e-34, 1e-30], device=a.device)[:, None]
    a[23, : K // 2], a[23, K // 2:] = a[23, : K // 2] * 1e-37, 0.0          # tiny ones alone, in some ranges nothing else
    a[24], a[25] = 2.0 ** -140, 0.0
    w[100:104] *= torch.tensor([1e35, 1e30, 1e20, 1e8], device=a.device)[:, None]
    w[104], w[105] = w[104] * 1e-35, 0.0
    a[40:42] *= 1e33
    w = w.as_subclass(type(ops.pack_weight(w)))
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    got, usual = (ops.linear(a, w, variant=v) for v in (plan(tile, ranges), 40))
    # (as for ordinary numbers; a product below 2^-126 rounds to 2^-149; rows of numbers below 2^-126 are what 32-bit instructions make of them)
    bound = 40 * U * size + K * 2.0 ** -149
    fits = size < 1e38
    fits[24] = False
    assert ((got.double() - want).abs() <= bound)[fits].all() and torch.equal(got.isfinite() | fits, usual.isfinite() | fits)
    assert torch.equal(got[24] == 0, usual[24] == 0) and ((got[24] - usual[24]).double().abs() <= bound[24]).all()
    assert (got[25] == 0).all() and (got[:, 105] == 0).all()


# 1.00389862 has the parts 1, 2^-8 and -2^-17: of such a product the parts left out are 2^-24, all of one sign
def test_products_whose_missing_parts_add_up():
    import torch
    M, N, K = 40, 200, 2048
    ops, a, w, _, _ = operands(M, N, K)
    x = 1 + 32704 * 2.0 ** -23
    a.fill_(x), w.fill_(x)
    for tile in range(TILES):
        for ranges in (1, 4):
            got = ops.linear(a, w, variant=plan(tile, ranges))
            # 2^-24, and as much again for the runs' sums, whose losses are made up for, and the last rounding
            assert ((got.double() / (K * x * x) - 1).abs() <= 2 * U).all()


def test_products_that_stay_with_the_32_bit_instructions():
    import torch
    from xyntetik_runner_amd.csrc.ops import F32Weight, load_ops
    ops, a, w, _, _ = operands(401, 4096, 1024)
    plain = w.as_subclass(torch.Tensor)                         # a matrix that is no model's weight
    assert torch.equal(ops.linear(a, plain), ops.linear(a, w, variant=40 + ops.lib.xr_f32_tile(401, 4096, 1024)))
    packed = ops.pack_weight(plain)
    assert isinstance(packed, F32Weight) and packed.data_ptr() == w.data_ptr() and type(packed[:5] * 2) is torch.Tensor
    assert torch.equal(ops.linear(a, packed), ops.linear(a, w)) and not torch.equal(ops.linear(a, packed), ops.linear(a, plain))
    take = ops.lib.xr_gemm_f32_parts_plan
    assert [take(*x) for x in ((16, 4096, 4096), (401, 4096, 448), (401, 4096, 4100), (401, 4096, 4128), (128, 3072, 768))] == [0] * 5
