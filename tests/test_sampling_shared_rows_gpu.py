"""Picks of rows that several workgroups share against the same picks by one workgroup a row: the tokens are equal."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rows(kind, W, V, rng):
    x = rng.standard_normal((W, V)).astype(np.float32) * 2.5
    if kind == "equal":
        x[:] = 1.25                                 # one bin holds the row: the general way
    elif kind == "steps":
        x = np.floor(x)                             # a few values, thousands of candidates each
    elif kind == "ruled_out":
        x[:, rng.permutation(V)[:V // 3]] = -np.inf
    elif kind == "near":
        x = 3.0 + x * 1e-8                          # z span less than the quick quotient is for
    elif kind == "far":
        x *= 1e19                                   # and logits beyond it
    elif kind == "peaked":
        x[np.arange(W), rng.integers(0, V, W)] = 60.0
    elif kind == "nothing":
        x[: W // 2] = -np.inf
        x[W // 2:, 5] = np.inf
    elif kind == "no_number":
        x[:, ::7] = np.nan
    return x


@pytest.mark.parametrize("kind", ["plain", "equal", "steps", "ruled_out", "near", "far", "peaked", "nothing", "no_number"])
@pytest.mark.parametrize("W,V", [(1, 8192), (3, 8195), (9, 32000), (64, 32001), (70, 16387)])
def test_shared_rows_pick_as_one_workgroup_does(kind, W, V):
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(W * 31 + V + len(kind))
    logits = torch.tensor(_rows(kind, W, V, rng), device=DEV)
    f = lambda v: torch.tensor(np.asarray(v, dtype=np.float32), device=DEV)
    i = lambda v: torch.tensor(np.asarray(v, dtype=np.int32), device=DEV)
    for turn in range(4):
        # greedy rows among them; cuts alone and together; a top-k of more candidates than a list holds; a draw at either end
        temp = rng.choice([0.0, 0.3, 0.8, 1.0, 1.3, 2e-7, 3e7], W, p=[.1, .2, .3, .15, .15, .05, .05])
        draw = rng.choice([0.0, 0.5, 1.0 - 2.0 ** -24, 0.123], W)
        top_k = rng.choice([0, 1, 40, 2048, 2049, 7000, V, V + 1], W) if turn else np.zeros(W)
        top_p = rng.choice([1.0, 0.95, 0.5, 0.0], W) if turn != 1 else np.ones(W)
        min_p = rng.choice([0.0, 0.05, 0.9, 1.0], W) if turn > 1 else np.zeros(W)
        args = f(temp), f(draw), i(top_k), f(top_p), f(min_p)
        shared = ops.sample(logits.clone(), args[0], args[1], top_k=args[2], top_p=args[3], min_p=args[4]).cpu().tolist()
        out = torch.empty((W,), dtype=torch.int32, device=DEV)
        one = logits.clone()
        ops.lib.check(ops.lib.xr_sample(out.data_ptr(), one.data_ptr(), W, V, V, args[0].data_ptr(), args[2].data_ptr(), args[3].data_ptr(),
                                        args[4].data_ptr(), None, args[1].data_ptr(), None, None, 0, None, 0, None,
                                        torch.cuda.current_stream().cuda_stream))
        assert shared == out.cpu().tolist(), (kind, W, V, turn)


@pytest.mark.parametrize("W", [1, 64])
def test_windows_of_a_batch(W):
    """A batch's recent tokens reach the kernels as they are kept: the picks are those with every row's penalty applied on the host."""
    from xyntetik_runner_amd.csrc.ops import load_ops
    from xyntetik_runner_amd.sampling import Sampler, SamplerState, SamplingParams
    rng = np.random.default_rng(W)
    V, rp = 9000, 1.5
    x = rng.standard_normal((W, V)).astype(np.float32) * 2
    want_x = x.copy()
    mk = lambda p: [SamplerState(SamplingParams(temperature=0.9, top_p=0.9, repeat_penalty=p, seed=r + 1)) for r in range(W)]
    states, plain = mk(rp), mk(1.0)
    for r, s in enumerate(states):
        recent = rng.integers(0, 60, int(rng.integers(1, 300))).tolist()
        for t in recent:
            s.accept(t)
        for t in recent[-256:]:
            v = want_x[r, t]
            want_x[r, t] = v / np.float32(rp) if v > 0 else v * np.float32(rp)
    sampler = Sampler(load_ops(), torch.device(DEV))
    got = sampler.sample(torch.tensor(x, device=DEV), states)
    assert got == sampler.sample(torch.tensor(want_x, device=DEV), plain)


# on either side of the lines between one workgroup a row, four of which the last picks, and eight that look for candidates; rows that are not 16-byte aligned
@pytest.mark.parametrize("kind", ["plain", "equal", "steps", "ruled_out", "near", "far", "peaked", "nothing", "no_number"])
@pytest.mark.parametrize("W,V,ld", [(2, 19996, 19996), (2, 20000, 20000), (64, 20004, 20008), (65, 20004, 20004), (3, 45996, 45996), (3, 46000, 46000), (2, 20001, 20003), (129, 46000, 46000)])
def test_ways_to_share_a_row_pick_alike(kind, W, V, ld):
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    assert {ops._sample_shares(w, v, a) for w, v, a in ((2, 19996, True), (65, 20004, True), (129, 46000, True))} == {(0, 0)}
    assert ops._sample_shares(64, 20004, True) == ops._sample_shares(3, 45996, True) == (4, 0)
    assert ops._sample_shares(3, 46000, True) == ops._sample_shares(2, 20001, False) == (8, 8)
    rng = np.random.default_rng(W * 31 + V + len(kind))
    room = torch.zeros((W, ld), device=DEV)
    room[:, :V] = torch.tensor(_rows(kind, W, V, rng), device=DEV)
    logits = room[:, :V]
    f = lambda v: torch.tensor(np.asarray(v, dtype=np.float32), device=DEV)
    i = lambda v: torch.tensor(np.asarray(v, dtype=np.int32), device=DEV)
    for turn in range(2):
        temp, draw = f(rng.choice([0.0, 0.3, 0.8, 1.3, 2e-7, 3e7], W, p=[.1, .25, .3, .25, .05, .05])), f(rng.choice([0.0, 0.5, 1.0 - 2.0 ** -24, 0.123], W))
        top_k, top_p, min_p = i(rng.choice([0, 1, 40, 2048, 2049, V], W)), f(rng.choice([1.0, 0.95, 0.0], W)), f(rng.choice([0.0, 0.05, 1.0], W) * turn)
        got = ops.sample(logits, temp, draw, top_k=top_k, top_p=top_p, min_p=min_p).cpu().tolist()
        out = torch.empty((W,), dtype=torch.int32, device=DEV)
        ops.lib.check(ops.lib.xr_sample(out.data_ptr(), logits.data_ptr(), W, V, ld, temp.data_ptr(), top_k.data_ptr(), top_p.data_ptr(), min_p.data_ptr(), None,
                                        draw.data_ptr(), None, None, 0, None, 0, None, torch.cuda.current_stream().cuda_stream))
        assert got == out.cpu().tolist(), (kind, W, V, turn)
