"""PolyNorm over rows kept in registers, either side of every length at which a row gets more lanes or more registers a lane."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import plain_suripel as S


@pytest.mark.parametrize("F", [4, 1020, 1024, 4092, 4096, 4100, 8192, 8196, 16384, 16388, 24576, 24580, 32768, 32772])
@pytest.mark.parametrize("T", [1, 70])
def test_polynorm_rows(F, T):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    z = (np.random.default_rng(F + T).normal(size=(T, F)) * 2).astype(np.float32)
    coef = torch.tensor([0.7, -1.3, 0.45, 0.2], device=dev)
    want = S.polynorm(z.astype(np.float64), coef.double().cpu().numpy(), 1e-5)
    t = torch.tensor(z, device=dev)
    # a value's four terms and three norms round to 2^-24 each, and a norm's sum of F squares adds some more
    bound = 2e-6 * np.abs(want).max()
    got = ops.polynorm(t, coef, 1e-5, torch.float32)
    assert np.abs(got.double().cpu().numpy() - want).max() < bound
    assert torch.equal(ops.polynorm(t, coef, 1e-5, torch.bfloat16), got.bfloat16())
    odd = torch.empty((T, F + 1), device=dev)       # rows that are not 16-byte aligned
    odd[:, 1:] = t
    assert np.abs(ops.polynorm(odd[:, 1:], coef, 1e-5, torch.float32).double().cpu().numpy() - want).max() < bound
    half = t.bfloat16()
    again = S.polynorm(half.double().cpu().numpy(), coef.double().cpu().numpy(), 1e-5)
    assert np.abs(ops.polynorm(half, coef, 1e-5, torch.bfloat16).double().cpu().numpy() - again).max() < np.abs(again).max() * 2.0 ** -8


@pytest.mark.parametrize("F", [8192, 8196, 16388, 24580, 32768])
def test_rows_on_either_side_of_one_a_compute_unit(F):
    """More than 256 long rows make their powers again: the same numbers, to a rounding of a term."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    z = torch.randn((257, F), device=dev) * 2
    coef = torch.tensor([0.7, -1.3, 0.45, 0.2], device=dev)
    few, many = ops.polynorm(z[:256], coef, 1e-5, torch.float32), ops.polynorm(z, coef, 1e-5, torch.float32)
    want = torch.tensor(S.polynorm(z.double().cpu().numpy(), coef.double().cpu().numpy(), 1e-5), device=dev)
    bound = 2e-6 * float(want.abs().max())          # (as above)
    assert float((many.double() - want).abs().max()) < bound and float((few.double() - want[:256]).abs().max()) < bound
