"""Products of few rows at the edges of their sizes: few weight rows, whose k-steps are taken in pairs by workgroups of 8 of them, and whole
steps of K, whose loads are a ring."""
import pytest

pytestmark = pytest.mark.gpu


# pairs: weight rows: fewer than a workgroup's 8, no multiple of 8 or 16, the most; columns: whole pairs of 32, an odd step at the end, a last step
# of 8.  Rings: one step, fewer than waves, fewer than a ring, one past it, waves with different numbers of steps; fewer than 4,096 weight
# rows, no multiple of 16, and more; 65,536 and more.  Batches (K no whole steps) beside them.
@pytest.mark.parametrize("N,K", [(7, 2048), (2048, 2048), (2041, 2080), (2024, 2056), (40, 14336), (1000, 4104), (2048, 10752),
                                 (40, 32), (3000, 288), (2060, 4128), (4100, 1056), (4112, 5152), (5000, 1064), (65552, 96), (65552, 2048),
                                 (3000, 2080), (6000, 2048), (4100, 512), (4100, 544)])
@pytest.mark.parametrize("M", [1, 7, 8, 9, 16])
def test_product(M, N, K):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a, w, bias, c = (torch.randn(s, generator=g, device=dev) for s in ((M, K + 8), (N, K), (N,), (M, N)))
    a, w = a.bfloat16()[:, 8:], (w * 0.1).bfloat16()
    want = a.double() @ w.double().T
    # exact products of bfloat16 numbers, at most K additions that round to 2^-24 of what has been added up so far
    bound = (K + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs() + c.double().abs())
    packed = ops.pack_weight(w)
    got = ops.linear(a, packed, out_dtype=torch.float32)
    assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(ops.linear(a, w, out_dtype=torch.float32), got)
    assert torch.equal(ops.linear(a, packed, bias=bias, out_dtype=torch.float32), got + bias)
    assert torch.equal(ops.linear(a, packed), got.bfloat16())
    out = c.clone()
    ops.linear(a, packed, out=out, accumulate=True)
    assert torch.equal(out, c + got)
    if N % 32 == 0 or N in (40, 4112, 3000):                    # and gated: the first rows' gate, the others' up rows
        F = N // 32 * 16
        gated = ops.linear_gated(a, ops.pack_weight(w[:2 * F].contiguous(), gated=True)).double()
        x, y = want[:, :F], want[:, F:2 * F]
        silu, room = x / (1 + torch.exp(-x)), bound[:, :F] + bound[:, F:2 * F]
        # (the sums' errors through the gate, whose slope is at most 1.1, and a bfloat16 rounding of 2^-9)
        assert ((gated - silu * y).abs() <= 1.1 * room * (1 + x.abs() + y.abs()) + 2.0 ** -8 * (silu * y).abs()).all()
    # a row's result does not depend on the rows beside it, on either side of 8 rows (from 65,536 weight rows on: on the same side, for more rows
    # are made in four waves and not in eight)
    few, most = (1, 16) if N < 65536 else (1, 8) if M <= 8 else (9, 16)
    assert torch.equal(ops.linear(a[:few], packed, out_dtype=torch.float32), got[:few])
    many = torch.cat([a, a[:1].expand(most - M, K)]) if M < most else a
    assert torch.equal(ops.linear(many.contiguous(), packed, out_dtype=torch.float32)[:M], got)


@pytest.mark.parametrize("N,K", [(40, 2048), (3000, 2048), (4112, 64)])
def test_rows_that_are_far_apart(N, K):
    """Rows that begin 2^28 numbers one behind the other: more bytes than 32 bits count."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    if torch.cuda.mem_get_info()[0] < 8 << 30:
        pytest.skip("nine such rows are 4.5 GiB")
    g = torch.Generator(device=dev)
    g.manual_seed(N + K)
    a, w = (torch.randn(s, generator=g, device=dev).bfloat16() for s in ((9, K), (N, K)))
    far = torch.empty((8 * 2 ** 28 + K,), dtype=torch.bfloat16, device=dev).as_strided((9, K), (2 ** 28, 1))
    far.copy_(a)
    want, bound = a.double() @ w.double().T, (K + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    for M in (8, 9):
        assert ((ops.linear(far[:M], ops.pack_weight(w), out_dtype=torch.float32).double() - want[:M]).abs() <= bound[:M]).all()


# (what reads them: a ring, batches, and batches with more than 256 partial sums)
@pytest.mark.parametrize("N,F,K", [(2048, 512, 2048), (2040, 8192, 2080), (24, 128256 // 16, 4096), (4104, 512, 512)])
@pytest.mark.parametrize("M", [1, 8, 9])
def test_the_norm_behind_it(M, N, F, K):
    """The product adds into a stream and leaves its weighted rows and the sums of their squares to the next product."""
    import torch
    from xyntetik_runner_amd.csrc.ops import UnscaledRows, load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a, w, x, nw, w2 = (torch.randn(s, generator=g, device=dev) for s in ((M, K), (N, K), (M, N), (N,), (F, N)))
    a, w, w2 = a.bfloat16(), ops.pack_weight((w * 0.05).bfloat16()), ops.pack_weight((w2 * 0.05).bfloat16())
    x = x * torch.linspace(0.1, 30, M, device=dev)[:, None]
    want = x.clone()
    ops.linear(a, w, out=want, accumulate=True)
    h = ops.linear_add_rmsnorm(a, w, x, nw, 1e-5, torch.bfloat16, defer=True)
    assert isinstance(h, UnscaledRows) and torch.equal(x, want) and torch.equal(h.data, (x * nw).bfloat16())
    d = x.double()
    # (sums of N squares, every one and every addition rounded to 2^-24)
    assert ((h.sumsq[:, :M].double().sum(0) - (d * d).sum(1)).abs() <= (N + 2) * 2.0 ** -24 * (d * d).sum(1)).all()
    scale = torch.rsqrt((d * d).mean(1, keepdim=True) + 1e-5)
    rows, wt = h.data.double() * scale, ops.linear(torch.eye(N, device=dev).bfloat16(), w2, out_dtype=torch.float32).double() if N % 8 == 0 else None
    got = ops.linear(h, w2, out_dtype=torch.float32).double()
    assert ((got - rows @ wt).abs() <= (N + 8) * 2.0 ** -23 * (rows.abs() @ wt.abs())).all()


def test_room_for_a_partial_sum_every_16_columns():
    """Room for half as many partial sums of squares as workgroups of 8 weight rows make: the kernel that needs no more."""
    import ctypes
    import torch
    from xyntetik_runner_amd.csrc.ops import XR_F32, _GemmNorm, _stream, load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    M, N, K = 3, 2048, 2048
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    a, w, x, nw = (torch.randn(s, generator=g, device=dev) for s in ((M, K), (N, K), (M, N), (N,)))
    a, w = a.bfloat16(), w.bfloat16()
    want, size = x.double() + a.double() @ w.double().T, x.double().abs() + a.double().abs() @ w.double().abs().T
    xg, sums = torch.empty((M, N), dtype=torch.bfloat16, device=dev), torch.full((N // 8, 16), -1.0, device=dev)
    then = _GemmNorm()
    then.norm_w, then.xg, then.ss_out, then.ss_out_rows = nw.data_ptr(), xg.data_ptr(), sums.data_ptr(), N // 16
    then.ss_inv_width, then.ss_eps = 1.0 / N, 1e-5
    ops.lib.check(ops.lib.xr_gemm_bf16(x.data_ptr(), a.data_ptr(), w.data_ptr(), None, M, N, K, K, N, XR_F32, 1, 0, 0.0, 0, 0,
                                       *ops._gemm_workspace(dev), ctypes.addressof(then), None, _stream()))
    assert then.ss_out_rows == N // 16 and (sums[N // 16:] == -1).all()
    assert ((x.double() - want).abs() <= (K + 4) * 2.0 ** -24 * size).all() and torch.equal(xg, (x * nw).bfloat16())
    d = x.double() ** 2
    assert ((sums[:N // 16, :M].double().sum(0) - d.sum(1)).abs() <= (N + 2) * 2.0 ** -24 * d.sum(1)).all()
