"""Layer norms to 32 bits with a row in registers and the norm with its convolution of four taps, either side of the widths at which
a lane gets more values: the fused kernel gives the bits of the two kernels it stands for, and both are the plain functions'."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import plain_suripel as S
from test_suripel_kernels_gpu import DEV, dev, step_ctx


@pytest.mark.parametrize("E", [6, 1023, 1024, 1030, 2048, 2049, 4096, 4100, 8192, 8193])
@pytest.mark.parametrize("B", [3, 130])
def test_layernorm_and_convolution(E, B):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(E + B)
    taps, n = 4, 3
    xs = rng.normal(size=(n, B, E)) * 2 + 0.3
    w, cw = rng.normal(size=E), rng.normal(size=(E, taps))
    hs = np.stack([S.layer_norm(dev(x).double().cpu().numpy(), dev(w).double().cpu().numpy(), 1e-5) for x in xs])
    slots = list(rng.permutation(B))
    st_a, st_b = (torch.zeros((B + 1, taps - 1, E), device=DEV) for _ in range(2))
    for t in range(n):
        ctx = step_ctx([t] * B, [1] * B, slots)
        x = dev(xs[t])
        two = ops.layernorm(x, dev(w), 1e-5, torch.float32)
        # mean, deviation and scaling round to 2^-24 of values up to 10 each
        assert np.abs(two.double().cpu().numpy() - hs[t]).max() < 5e-6 * np.abs(hs[t]).max()
        two = ops.causal_conv(two, dev(cw), st_b, ctx, torch.float32, residual=True)
        got = ops.layernorm_conv(x, dev(w), 1e-5, dev(cw), st_a, ctx, torch.float32)
        if B <= 128:            # (the fused kernel and a norm of more rows add with other numbers of waves)
            assert torch.equal(got, two) and torch.equal(st_a, st_b)
        want = hs[t] + sum(cw.astype(np.float32)[:, taps - 1 - k] * hs[t - k] for k in range(min(t, taps - 1) + 1))
        assert np.abs(got.double().cpu().numpy() - want).max() < 1e-5 * np.abs(want).max()
        assert torch.equal(st_a[torch.tensor(slots, device=DEV), -1], got.new_tensor(0) + ops.layernorm(x, dev(w), 1e-5, torch.float32)) or B > 128
