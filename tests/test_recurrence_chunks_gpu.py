"""Retention and the gated delta rule in chunks of 64 rows, against the recurrences run token by token in 64 bits: portions
that end within a chunk, on its edge and one row past it, beside short requests and decoded tokens; decays of one, near
nothing and nothing; errors no larger than those of the kernel that goes token by token."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import plain_suripel as S
from test_suripel_kernels_gpu import DEV, dev, step_ctx


def run(ops, kind, qs, ks, vs, extra, H, G, D, Dv, plans, slots, n_slots, activation=None, k_scale=1.0):
    import torch
    state = torch.full((n_slots + 1,) + tuple(ops.recurrence_state_shape(H, D, Dv)), float("nan"), device=DEV)
    state[torch.tensor(slots, device=DEV)] = 0
    got = [np.zeros((len(q), H, Dv)) for q in qs]
    plans = [list(p) for p in plans]
    while any(plans):
        live = [b for b in range(len(qs)) if plans[b]]
        parts = [plans[b].pop(0) for b in live]
        ctx = step_ctx([p[0] for p in parts], [p[1] for p in parts], [slots[b] for b in live])
        cat = lambda xs: np.concatenate([xs[b][i:i + n].reshape(n, -1) for b, (i, n) in zip(live, parts)])
        row = dev(np.concatenate([cat(qs), cat(ks), cat(vs), np.zeros((ctx.T, 4))], axis=1))
        q, k, v = row[:, :G * D], row[:, G * D:2 * G * D], row[:, 2 * G * D:2 * G * D + H * Dv]
        if kind == "delta":
            gates = dev(np.concatenate([cat(extra[0]), cat(extra[1])], axis=1))
            o = ops.linear_recurrence("delta", q, k, v, state, ctx, H, G, D, Dv, beta=gates[:, :H], gate=gates[:, H:])
        else:
            o = ops.linear_recurrence("retention", q, k, v, state, ctx, H, G, D, Dv, decay=dev(extra), activation=activation, k_scale=k_scale)
        o = o.cpu().numpy()
        r = 0
        for b, (i, n) in zip(live, parts):
            got[b][i:i + n] = o[r:r + n].reshape(n, H, Dv)
            r += n
    assert torch.isnan(state[n_slots]).all(), "the row that is nobody's was written"
    return got


def error(got, want):
    return max(np.abs(g - w).max() / np.abs(w).max() for g, w in zip(got, want))


PORTIONS = [[(0, 64), (64, 65), (129, 1), (130, 200)], [(0, 63), (63, 1), (64, 2)], [(0, 127), (127, 128)], [(0, 1), (1, 70)]]


def both(ops, monkeypatch, *args, **kw):
    """(in chunks from portions of ``shortest`` rows on, token by token)"""
    shortest = kw.pop("shortest", 1)
    monkeypatch.setattr(type(ops), "CHUNKS_FROM", 1)
    monkeypatch.setattr(type(ops), "chunked_rows", lambda self, kind, q_lens, H, Dv: shortest if max(q_lens) >= shortest else None)
    chunks = run(ops, *args, **kw)
    monkeypatch.setattr(type(ops), "CHUNKS_FROM", 1 << 30)
    plain = run(ops, *args, **kw)
    monkeypatch.undo()
    return chunks, plain


@pytest.mark.parametrize("H,G,D,Dv", [(2, 2, 48, 16), (4, 2, 64, 32), (2, 1, 80, 48), (2, 2, 96, 16), (1, 1, 112, 64), (4, 2, 128, 128)])
def test_delta_rule_in_chunks(monkeypatch, H, G, D, Dv):
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(D + Dv)
    lens = [sum(n for _, n in p) for p in PORTIONS]
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    qs = [f32(S.unit(rng.normal(size=(n, G, D))) * D ** -0.5) for n in lens]
    ks = [f32(S.unit(rng.normal(size=(n, G, D)) + 0.5)) for n in lens]          # (keys that have much in common)
    vs = [f32(rng.normal(size=(n, H, Dv))) for n in lens]
    beta = [f32(S.sigmoid(rng.normal(size=(n, H)) * 2 + 1)) for n in lens]
    g = [f32(np.exp(-rng.exponential(0.1, size=(n, H)))) for n in lens]
    g[0][70:75] = 0.0                           # a state that is gone
    g[1][:] = 1.0
    g[2][100] = 1e-38
    rep = H // G
    want = [S.gated_delta_rule(np.repeat(q, rep, 1), np.repeat(k, rep, 1), v, b, gg) for q, k, v, b, gg in zip(qs, ks, vs, beta, g)]
    chunks, plain = both(ops, monkeypatch, "delta", qs, ks, vs, (beta, g), H, G, D, Dv, PORTIONS, [2, 0, 4, 1], 5)
    # a row is a sum of some D products with a state that up to 330 updates rounded, 2^-24 each: 5e-6 of the largest value
    assert error(chunks, want) < 5e-6, (error(chunks, want), error(plain, want))
    assert error(chunks, want) < 2 * error(plain, want) + 2e-7, (error(chunks, want), error(plain, want))


@pytest.mark.parametrize("kind", ["delta", "retention"])
@pytest.mark.parametrize("shortest", [2, 64, 65, 200])
def test_long_portions_in_chunks_beside_short_ones_token_by_token(monkeypatch, kind, shortest):
    """One step's requests go both ways, each once: the portions of ``shortest`` rows and more in chunks, the others token by token,
    in whatever order they come."""
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    H, D, Dv = 4, 64, 32
    rng = np.random.default_rng(shortest)
    lens = [sum(n for _, n in p) for p in PORTIONS]
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    qs, ks = ([f32(S.unit(rng.normal(size=(n, H, D)))) for n in lens] for _ in range(2))
    vs = [f32(rng.normal(size=(n, H, Dv))) for n in lens]
    if kind == "delta":
        extra = ([f32(S.sigmoid(rng.normal(size=(n, H)))) for n in lens], [f32(np.exp(-rng.exponential(0.1, size=(n, H)))) for n in lens])
        want = [S.gated_delta_rule(q, k, v, b, g) for q, k, v, b, g in zip(qs, ks, vs, *extra)]
    else:
        extra = f32(np.array([0.97, 1.0, 0.5, 0.9]))
        want = [S.retention(q, k, v, extra) for q, k, v in zip(qs, ks, vs)]
    mixed, plain = both(ops, monkeypatch, kind, qs, ks, vs, extra, H, H, D, Dv, PORTIONS, [2, 0, 4, 1], 5, shortest=shortest)
    assert error(mixed, want) < 5e-6, (error(mixed, want), error(plain, want))


@pytest.mark.parametrize("H,D,Dv", [(2, 48, 16), (3, 64, 32), (1, 80, 48), (2, 128, 128)])
@pytest.mark.parametrize("activation", [None, "silu"])
def test_retention_in_chunks(monkeypatch, H, D, Dv, activation):
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(D + Dv)
    lens = [sum(n for _, n in p) for p in PORTIONS]
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    qs, ks = ([f32(rng.normal(size=(n, H, D))) for n in lens] for _ in range(2))
    vs = [f32(rng.normal(size=(n, H, Dv))) for n in lens]
    decay = f32(np.array([0.97, 1.0, 0.0][:H]))
    act = S.silu if activation else (lambda x: x)
    want = [S.retention(act(q), act(k) * 0.25, act(v), decay) for q, k, v in zip(qs, ks, vs)]
    chunks, plain = both(ops, monkeypatch, "retention", qs, ks, vs, decay, H, H, D, Dv, PORTIONS, [2, 0, 4, 1], 5, activation=activation, k_scale=0.25)
    assert error(chunks, want) < 5e-6, (error(chunks, want), error(plain, want))
    assert error(chunks, want) < 2 * error(plain, want) + 2e-7, (error(chunks, want), error(plain, want))


@pytest.mark.parametrize("kind,H,G,D,Dv", [("delta", 2, 2, 64, 32), ("delta", 2, 1, 128, 64), ("retention", 2, 2, 64, 32), ("retention", 2, 2, 128, 64)])
@pytest.mark.parametrize("decay,common", [(0.1, 0.5), (0.1, 0.0), (0.003, 0.0)])
def test_errors_are_no_larger_than_token_by_token(monkeypatch, kind, H, G, D, Dv, decay, common):
    """Over portions of some hundred rows, in the 2-norm."""
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    rng = np.random.default_rng(D + int(1000 * decay) + int(10 * common))
    portions = [[(0, 700)], [(0, 200), (200, 300)]]
    lens = [700, 500]
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    vs = [f32(rng.normal(size=(n, H, Dv))) for n in lens]
    qs, ks = ([f32(S.unit(rng.normal(size=(n, G, D)) + c)) for n in lens] for c in (0.0, common))
    if kind == "delta":
        extra = ([f32(S.sigmoid(rng.normal(size=(n, H)) * 2 + 1)) for n in lens], [f32(np.exp(-rng.exponential(decay, size=(n, H)))) for n in lens])
        want = [S.gated_delta_rule(np.repeat(q, H // G, 1), np.repeat(k, H // G, 1), v, b, g) for q, k, v, b, g in zip(qs, ks, vs, *extra)]
    else:
        extra = f32(np.array([1.0 - decay, 1.0]))
        want = [S.retention(q, k, v, extra) for q, k, v in zip(qs, ks, vs)]
    chunks, plain = both(ops, monkeypatch, kind, qs, ks, vs, extra, H, G, D, Dv, portions, [1, 0], 3)
    off = lambda got: np.sqrt(sum(((g - w) ** 2).sum() for g, w in zip(got, want)) / sum((w ** 2).sum() for w in want))
    # (two roundings of the same size, met in another order: a tenth for chance; in single 32-bit chains it was 1.4 to 2.3 for the delta rule)
    assert off(chunks) <= 1.1 * off(plain), (off(chunks), off(plain))


def test_which_steps_read_rows_again():
    """Where retention applies its activation to the rows before the recurrence instead of in it."""
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops = load_ops()
    again = lambda kind, D, *q_lens: ops.recurrence_reads_rows_again(kind, step_ctx([0] * len(q_lens), list(q_lens), list(range(len(q_lens)))), 32, D, 128)
    assert again("retention", 128, 1, 200, 1) and again("retention", 128, 1023) and again("retention", 256, 1024)
    assert not again("retention", 128, 95) and not again("retention", 128, *[100] * 20) and not again("retention", 256, 1023)


@pytest.mark.parametrize("kind,G,D", [("retention", 24, 48), ("retention", 24, 64), ("retention", 24, 80), ("delta", 12, 48)])
@pytest.mark.parametrize("activation", [None, "silu"])
def test_more_workgroups_than_compute_units(monkeypatch, kind, G, D, activation):
    """Small heads of several portions at once, 288 workgroups, whose operands go through LDS; without an activation the last step's 144 and the 72 of a portion go straight to registers.
    A decay below zero, and then an infinity in a value: those columns come out as token by token."""
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, H, Dv = load_ops(), 24, 48
    rng = np.random.default_rng(D + G)
    lens = [sum(n for _, n in p) for p in PORTIONS]
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    qs, ks = ([f32(S.unit(rng.normal(size=(n, G, D)))) for n in lens] for _ in range(2))
    vs = [f32(rng.normal(size=(n, H, Dv))) for n in lens]
    if kind == "delta":
        if activation:
            pytest.skip("the delta rule's activation is its convolution's")
        extra = ([f32(S.sigmoid(rng.normal(size=(n, H)))) for n in lens], [f32(np.exp(-rng.exponential(0.1, size=(n, H)))) for n in lens])
        want = [S.gated_delta_rule(np.repeat(q, 2, 1), np.repeat(k, 2, 1), v, b, g) for q, k, v, b, g in zip(qs, ks, vs, *extra)]
    else:
        extra = f32(np.resize([0.97, 1.0, 0.0, 0.5, -0.5], H))
        act = S.silu if activation else (lambda x: x)
        want = [S.retention(act(q), act(k) * 0.25, act(v), extra) for q, k, v in zip(qs, ks, vs)]
    kw = dict(activation=activation, k_scale=0.25) if kind == "retention" else {}
    chunks, plain = both(ops, monkeypatch, kind, qs, ks, vs, extra, H, G, D, Dv, PORTIONS, [2, 0, 4, 1], 5, **kw)
    # as above: 2^-24 of each of some 330 updates of a state
    assert error(chunks, want) < 5e-6, (error(chunks, want), error(plain, want))
    assert error(chunks, want) < 2 * error(plain, want) + 2e-7, (error(chunks, want), error(plain, want))
    vs[0][30, 3, 5] = np.inf
    broken, plain = both(ops, monkeypatch, kind, qs, ks, vs, extra, H, G, D, Dv, PORTIONS, [2, 0, 4, 1], 5, **kw)
    for b, p, c in zip(broken, plain, chunks):
        assert np.array_equal(np.isfinite(b), np.isfinite(p))
    assert np.array_equal(broken[0][:30], chunks[0][:30]) or error([broken[0][:30]], [chunks[0][:30]]) < 1e-6
    assert not np.isfinite(broken[0][30:, 3, 5]).any() and np.isfinite(broken[1]).all()
