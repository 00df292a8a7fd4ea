"""Layer norm and convolution of steps of several rows a request, in one kernel and in two: rows on either side of a workgroup's blocks,
portions shorter than the carried inputs, and the carried inputs after each portion."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import plain_suripel as S
from test_suripel_kernels_gpu import DEV, dev, step_ctx

# rows a request brings in three steps (0 rows: it is not there), blocks of 5 and of 8 rows
PORTIONS = [([4], [5], [6]), ([1, 2, 5, 6, 7], [3, 1, 10, 4, 1], [2, 16, 1, 15, 8]), ([9, 3, 1] + [1] * 70, [2, 8, 17] + [1] * 69 + [2], [1, 1, 40] + [2] * 70),
            ([133], [2], [7])]


@pytest.mark.parametrize("E", [4, 252, 2048, 2052, 4096])
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("portions", PORTIONS, ids=lambda p: f"{len(p[0])}x{p[0][0]}")
def test_norm_and_convolution(portions, taps, E):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    B = len(portions[0])
    if B > 8 and E > 2052:
        pytest.skip("many requests at small widths only")
    rng = np.random.default_rng(E + B + taps)
    f32 = lambda a: a.astype(np.float32).astype(np.float64)
    weight = rng.normal(size=E) if taps != 3 else None
    cw, slots = f32(rng.normal(size=(E, taps))), list(rng.permutation(B + 3)[:B])
    states = [torch.zeros((B + 4, taps - 1, E), device=DEV) for _ in range(2)]
    carried, at = np.zeros((B, taps - 1, E)), [0] * B
    for lens in portions:
        ctx = step_ctx(at, lens, slots)
        x = f32(rng.normal(size=(sum(lens), E + 4)) * 2 + 0.3)
        xd = dev(x)[:, :E]
        w = dev(weight) if weight is not None else None
        half = ops.layernorm_conv_rows(xd, w, 1e-5, dev(cw), states[0].clone(), ctx, torch.bfloat16)
        got = ops.layernorm_conv_rows(xd, w, 1e-5, dev(cw), states[0], ctx, torch.float32)
        assert got is not None
        two = ops.causal_conv(ops.layernorm(xd, w, 1e-5, torch.float32), dev(cw), states[1], ctx, torch.float32, residual=True)
        h = S.layer_norm(x[:, :E], f32(weight) if weight is not None else np.ones(E), 1e-5)
        row, want = 0, np.empty_like(h)
        for b, n in enumerate(lens):
            seen = np.concatenate([carried[b], h[row:row + n]])
            want[row:row + n] = h[row:row + n] + sum(cw[:, j] * seen[j:j + n] for j in range(taps))
            carried[b] = seen[len(seen) - (taps - 1):]
            row += n
        # a norm's rounding (2^-24 of values up to 10) through up to four products; the carried inputs are norms
        scale = np.abs(want).max()
        for y in (got, two):
            assert np.abs(y.double().cpu().numpy() - want).max() < 1e-5 * scale
        for st in states:
            assert np.abs(st[torch.tensor(slots, device=DEV)].double().cpu().numpy() - carried).max() < 5e-6 * np.abs(h).max()
            untouched = [i for i in range(B + 4) if i not in slots]
            assert not st[torch.tensor(untouched, device=DEV)].any()
        states[1].copy_(states[0])
        at = [a + n for a, n in zip(at, lens)]
        # two results rounded to bfloat16 from the same 32 bits differ nowhere
        assert torch.equal(half, got.bfloat16())


@pytest.mark.parametrize("taps", [1, 3, 4, 5, 9, 10, 16])
@pytest.mark.parametrize("dtypes", ["float32 float32", "float32 bfloat16", "bfloat16 bfloat16"])
def test_convolution_of_portions(dtypes, taps):
    """Nine taps are the most whose state one block of a request reads; ten go to the kernel that moves states on."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    tu, to = (getattr(torch, d) for d in dtypes.split())
    rng = np.random.default_rng(taps)
    C = 300
    for portions in PORTIONS[1:]:
        B = len(portions[0])
        cw, bias, slots = dev(rng.normal(size=(C, taps))), dev(rng.normal(size=C)), list(rng.permutation(B + 2)[:B])
        state = torch.zeros((B + 3, taps - 1, C), device=DEV, dtype=tu) if taps > 1 else None
        carried, at = np.zeros((B, taps - 1, C)), [0] * B
        for lens in portions:
            ctx = step_ctx(at, lens, slots)
            u = dev(rng.normal(size=(sum(lens), C + 1))).to(tu)[:, :C]
            got = ops.causal_conv(u, cw, state, ctx, to, activation="silu", bias=bias).double().cpu().numpy()
            h, w, bb = u.double().cpu().numpy(), cw.double().cpu().numpy(), bias.double().cpu().numpy()
            row, want = 0, np.empty_like(h)
            for b, n in enumerate(lens):
                seen = np.concatenate([carried[b], h[row:row + n]])
                y = bb + sum(w[:, j] * seen[j:j + n] for j in range(taps))
                want[row:row + n] = y / (1 + np.exp(-y))
                carried[b] = seen[len(seen) - (taps - 1):]
                row += n
            # 32-bit sums of up to 17 terms; a result in bfloat16 is half an ulp off
            assert np.abs(got - want).max() < (1e-5 if to == torch.float32 else 2.0 ** -8) * np.abs(want).max()
            if taps > 1:
                assert np.array_equal(state[torch.tensor(slots, device=DEV)].double().cpu().numpy(), carried)
            at = [a + n for a, n in zip(at, lens)]
