"""32-bit products of a few rows that norm their rows or gate their result themselves, against 64 bits and the kernels one by one."""
import pytest

pytestmark = pytest.mark.gpu


# rows: one, few, the most; outputs: fewer than a workgroup makes, no multiple of it, past the lines between 2 and 4 or 8 weight rows a
# wave; columns: less than a wave's 256, no multiple of them, several
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(1, 4), (7, 64), (176, 64), (250, 260), (4100, 512), (16390, 256), (8200, 4096)])
def test_normed_and_gated(M, N, K):
    import torch
    from xyntetik_runner_amd.csrc.ops import UnnormedRows, load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(M * 7 + N + K)
    x, w, bias = (torch.randn(s, generator=g, device=dev) for s in ((M, K + 4), (2 * N, K), (2 * N,)))
    x = x[:, :K]                                            # rows that are part of wider ones
    wn = torch.rand(K, generator=g, device=dev) + 0.5
    h64 = x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * wn.double()
    h = UnnormedRows(x, wn, 1e-5)
    # every product and sum rounds to 2^-24 of what has been added up so far, the norm's factor and weight a few times more
    size = h64.abs() @ w.double().abs().T + bias.double().abs()
    bound, want = (K + 12) * 2.0 ** -24 * size, h64 @ w.double().T + bias.double()
    got = ops.linear(h, w, bias=bias)
    assert ((got.double() - want).abs() <= bound).all()
    assert ((ops.linear(h, w[:N]).double() - h64 @ w[:N].double().T).abs() <= bound[:, :N]).all()
    gate, up = want[:, :N], want[:, N:]
    silu = gate / (1 + torch.exp(-gate))
    # (the gate's derivative is at most 1.1, its value at most |gate|)
    room = 1.1 * bound[:, :N] * up.abs() + silu.abs() * bound[:, N:] + bound[:, :N] * bound[:, N:] + 2.0 ** -20 * (silu * up).abs()
    assert ((ops.linear_gated(h, w, bias=bias).double() - silu * up).abs() <= room).all()
    # rows that are normed already: the same bits as the product and the gate's kernel one after the other
    rows = ops.rmsnorm(x, wn, 1e-5, torch.float32)
    for act, param in (("silu", 0.0), ("clamped_swish", 7.0)):
        assert torch.equal(ops.linear_gated(rows, w, bias=bias, activation=act, param=param),
                           ops.gate_mul(ops.linear(rows, w, bias=bias), act, param))
    # where a product cannot norm its rows the norm's kernel does
    out = torch.randn(M, 2 * N, generator=g, device=dev)
    base = out.clone()
    ops.linear(h, w, out=out, accumulate=True)
    assert torch.equal(out, base + ops.linear(rows, w))


def test_more_rows_are_normed_by_the_norms_kernel():
    import torch
    from xyntetik_runner_amd.csrc.ops import UnnormedRows, load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    torch.manual_seed(5)
    for M in (ops.EXTRA_ROWS, ops.EXTRA_ROWS + 1):
        a, w, x, wn = (torch.randn(s, device=dev) for s in ((M, 64), (96, 64), (M, 96), (96,)))
        got = ops.linear_add_rmsnorm(a, w, x, wn, 1e-5, torch.float32, defer=True)
        assert isinstance(got, UnnormedRows) == (M <= ops.EXTRA_ROWS)
        assert not isinstance(ops.linear_add_rmsnorm(a, w, x, wn, 1e-5, torch.float32), UnnormedRows)      # not asked for


# one row and the most, and outputs with 2, 4 and 8 weight rows a wave
@pytest.mark.parametrize("M", [1, 3, 4])
@pytest.mark.parametrize("N,K", [(64, 176), (252, 260), (16388, 256), (8192, 4096), (16384, 4096)])
def test_deferred_rows_stay_what_they_are_when_the_stream_is_written_again(M, N, K):
    """What comes back is a copy: a part may add to the stream between two products of the rows it was given."""
    import torch
    from xyntetik_runner_amd.csrc.ops import UnnormedRows, load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a, w, x, bias, w2 = (torch.randn(s, generator=g, device=dev) for s in ((M, K), (N, K), (M, N + 4), (N,), (96, N)))
    x, wn = x[:, 4:], torch.rand(N, generator=g, device=dev) + 0.5               # (a stream that is part of wider rows)
    want = x.clone()
    ops.linear(a, w, bias=bias, out=want, accumulate=True)
    h = ops.linear_add_rmsnorm(a, w, x, wn, 1e-5, torch.float32, bias=bias, defer=True)
    assert isinstance(h, UnnormedRows)
    assert torch.equal(x, want) and torch.equal(h.data, want)                    # the bits that the plain sum leaves
    first, gated = ops.linear(h, w2), ops.linear_gated(h, w2)
    ops.linear(a, w, out=x, accumulate=True)
    assert not torch.equal(x, want)
    assert torch.equal(ops.linear(h, w2), first) and torch.equal(ops.linear_gated(h, w2), gated)
