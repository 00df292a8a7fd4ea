"""One kernel for a decoded token of a recurrence, and one for a convolution and the store behind it, against the kernels they stand for."""
import types

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ctx_of(B, t, slots, tables=None):
    i = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    c = types.SimpleNamespace(B=B, T=B, max_q_len=1, q_lens=[1] * B, cu_q=i(list(range(B + 1))), slots=i(slots), req_of_token=i(list(range(B))),
                              positions=i([t + 3 * b for b in range(B)]), starts=[t + 3 * b for b in range(B)])
    c.starts_dev = c.positions
    c.block_table = lambda group: i(tables)
    return c


def near(got, want, what):
    """32-bit sums of up to 128 terms in another order: 4e-6 of the largest; of results in bfloat16 an ulp where they round apart."""
    tol = 4e-6 if got.dtype == torch.float32 else 2.0 ** -7
    got, want = got.double(), want.double()
    assert torch.isfinite(got).all() and float((got - want).abs().max()) <= tol * float(want.abs().max()), what


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,Dv,weight", [(2, 2, 33, 1, 0), (4, 2, 48, 70, 1), (3, 1, 64, 128, 2), (2, 1, 127, 65, 1), (4, 2, 128, 128, 1), (5, 5, 128, 64, 0)])
@pytest.mark.parametrize("kind", ["delta", "retention"])
def test_one_kernel_a_token(kind, H, G, D, Dv, weight, dtype):
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    if kind == "retention":
        G = H
    rng = np.random.default_rng(H * 1000 + D + Dv)
    f = lambda x: torch.tensor(np.asarray(x, dtype=np.float32), device=DEV)
    B, slots = 3, [2, 0, 3]
    states = [torch.zeros((5,) + tuple(ops.recurrence_state_shape(H, D, Dv)), device=DEV) for _ in range(2)]
    # D is more than 32, so a column lies in 16 lanes; the rows past D stay zero
    w = [None, f(rng.normal(size=Dv)), f(rng.normal(size=H * Dv))][weight]
    a_log, dt_bias, decay = f(rng.normal(size=H)), f(rng.normal(size=H)), f(rng.uniform(0.7, 1.0, size=H))
    rot = 0 if D % 2 or kind == "delta" else D if D < 128 else 96
    inv = f(10000.0 ** (-np.arange(rot // 2) / max(1, rot // 2))) if rot else None
    act = ["silu", "sigmoid"][D % 2]
    for t in range(4):
        ctx = ctx_of(B, 1000 * t, slots)
        row = f(rng.normal(size=(B, 2 * G * D + 2 * H * Dv + 2 * H + 5)))
        part = lambda x: (x[:, :G * D], x[:, G * D:2 * G * D], x[:, 2 * G * D:2 * G * D + H * Dv])
        rest = row[:, 2 * G * D + H * Dv:]
        gate, b, a = rest[:, :H * Dv], rest[:, H * Dv:H * Dv + H], rest[:, H * Dv + H:H * Dv + 2 * H]
        common = dict(gate_activation=act)
        if kind == "delta":
            got = ops.recurrence_step("delta", *part(row), states[0], ctx, H, G, D, Dv, gate, w, 1e-5, dtype, beta=b, gate=a, a_log=a_log,
                                      dt_bias=dt_bias, q_scale=D ** -0.5, unit_eps=1e-6, **common)
        else:
            got = ops.recurrence_step("retention", *part(row), states[0], ctx, H, G, D, Dv, gate, w, 1e-5, dtype, decay=decay, inv_freq=inv, rot=rot,
                                      k_scale=D ** -0.5, **common)
        q, k, v = part(row)
        if kind == "delta":
            ops.delta_prepare_(q, k, b, a, a_log, dt_bias, G, H, D, D ** -0.5, 1e-6)
            o = ops.linear_recurrence("delta", q, k, v, states[1], ctx, H, G, D, Dv, beta=b, gate=a)
        else:
            ops.rotate_rows_(q, ctx.positions, inv, H, D, rot, 1.0)
            ops.rotate_rows_(k, ctx.positions, inv, H, D, rot, D ** -0.5)
            o = ops.linear_recurrence("retention", q, k, v, states[1], ctx, H, H, D, Dv, decay=decay)
        want = ops.gated_rmsnorm(o, gate, w, H, Dv, 1e-5, dtype, gate_activation=act)
        near(got, want, f"token {t}")
        near(states[0], states[1], f"state {t}")
        assert not states[0][1].any() and not states[0][4].any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,Hk,D,Dv,taps,ps", [(3, 1, 7, 5, 2, 16), (8, 2, 128, 128, 4, 64), (4, 0, 64, 64, 4, 64), (2, 2, 48, 96, 16, 32)])
def test_convolution_and_store(H, Hk, D, Dv, taps, ps, dtype):
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(D + taps)
    f = lambda x: torch.tensor(np.asarray(x, dtype=np.float32), device=DEV)
    B, slots, Q, K = 3, [2, 0, 3], H * D, Hk * D
    C = Q + Hk * (D + Dv)
    w = f(rng.normal(size=(C, taps)))
    tables = [[3, 1], [2, 6], [4, 5]]
    mk = lambda: (torch.zeros((5, taps - 1, C), device=DEV), torch.zeros((7, max(Hk, 1), ps, D), dtype=dtype, device=DEV),
                  torch.zeros((7, max(Hk, 1), Dv, ps), dtype=dtype, device=DEV))
    one, two = mk(), mk()
    for t in range(ps - 7, ps + 3):
        ctx = ctx_of(B, t, slots, tables)
        u = f(rng.normal(size=(B, C + 3)))[:, :C]
        got = ops.conv_qkv_store(u, w, one[0], one[1] if Hk else None, one[2] if Hk else None, ctx, 0, H, Hk, D, Dv, ps, dtype)
        y = ops.causal_conv(u, w, two[0], ctx, torch.float32)
        want = ops.qkv_store(y[:, :Q], y[:, Q:Q + K] if Hk else None, y[:, Q + K:] if Hk else None, two[1], two[2], ctx, 0, H, Hk, D, Dv, ps, dtype)
        assert torch.equal(got, want)
        assert all(torch.equal(a, b) for a, b in zip(one, two))
