"""The sampled pick over long rows (histogram, one bin gathered and sorted a cut) against a sort of the whole row: rows whose
cuts fall where the bins end, into bins that do not fit the list, behind masked logits and among ties; the entry point that
shares a row out and the one that does not give the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pick(row, temp, draw, top_k, top_p, min_p):
    """By a stable sort in 64 bits: z descending, then id ascending."""
    z = (row / np.float32(temp)).astype(np.float64)
    order = np.argsort(-np.where(np.isnan(z), -np.inf, z), kind="stable")
    order = order[~np.isnan(z[order])]
    if len(order) == 0 or not np.isfinite(z[order[0]]):
        return 0
    if 0 < top_k < len(row):
        order = order[:top_k]
    p = np.exp(z[order] - z[order[0]])
    if top_p < 1.0:
        n = int(np.searchsorted(np.cumsum(p), top_p * p.sum())) + 1
        order, p = order[:n], p[:n]
    keep = p >= min_p
    order, p = order[keep], p[keep]
    return int(order[min(int(np.searchsorted(np.cumsum(p), draw * p.sum(), side="right")), len(order) - 1)])


def rows_of(kind, V, rng):
    row = (rng.standard_normal(V) * 2.5).astype(np.float32)
    if kind == "flat":                      # every bin holds more than the list; the cuts go the general way
        row[:] = rng.integers(0, 3, V).astype(np.float32) * 1e-3
    elif kind == "equal":
        row[:] = 1.25
    elif kind == "masked":                  # most of the vocabulary ruled out
        row[rng.random(V) < 0.97] = -np.inf
    elif kind == "ties":                    # thousands of equal candidates at the cut
        row[:] = np.round(row * 2) / 2
    elif kind == "peaked":
        row[V - 3] = 30.0
    elif kind == "nan":
        row[::7] = np.nan
    elif kind == "nothing":
        row[:] = -np.inf
    return row


@pytest.mark.parametrize("V", [8192, 8195, 50021, 128256])
def test_pick_by_bins(V):
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    rng = np.random.default_rng(V)
    rows, opts = [], []
    for kind in ("normal", "flat", "equal", "masked", "ties", "peaked", "nan", "nothing"):
        for top_k, top_p, min_p in ((0, 1.0, 0.0), (1, 1.0, 0.0), (40, 0.9, 0.05), (2048, 0.95, 0.0), (2049, 1.0, 0.0), (V - 1, 0.8, 0.0),
                                    (0, 0.95, 0.0), (0, 0.0, 0.0), (0, 1.0, 0.02), (0, 0.9, 1.0), (V + 5, 0.999, 1e-6)):
            rows.append(rows_of(kind, V, rng))
            draw = float(rng.integers(0, 1 << 24)) / (1 << 24)
            opts.append((float(rng.choice([0.3, 0.8, 1.3])), draw, top_k, float(np.float32(top_p)), float(np.float32(min_p))))
    f = lambda i: torch.tensor([o[i] for o in opts], dtype=torch.float32, device=dev)
    top_k = torch.tensor([o[2] for o in opts], dtype=torch.int32, device=dev)
    logits = torch.tensor(np.stack(rows), device=dev)
    before = logits.clone()
    got = ops.sample(logits, f(0), f(1), top_k=top_k, top_p=f(3), min_p=f(4)).cpu().tolist()
    want = [pick(r, *o) for r, o in zip(rows, opts)]
    assert [(i, g) for i, g in enumerate(got) if g != want[i]] == [(i, w) for i, w in enumerate(want) if w != got[i]], opts
    assert torch.equal(logits.view(torch.int32), before.view(torch.int32))
    # a row whose address allows no 16-byte loads, and one row alone
    odd = torch.empty((len(rows), V + 1), device=dev)
    odd[:, 1:] = logits
    assert ops.sample(odd[:, 1:], f(0), f(1), top_k=top_k, top_p=f(3), min_p=f(4)).cpu().tolist() == got
    assert ops.sample(logits[:1], f(0)[:1], f(1)[:1], top_k=top_k[:1], top_p=f(3)[:1], min_p=f(4)[:1]).cpu().tolist() == got[:1]
    # without options: no work area, one workgroup a row does it all
    plain = ops.sample(logits, f(0), f(1)).cpu().tolist()
    assert plain == [pick(r, o[0], o[1], 0, 1.0, 0.0) for r, o in zip(rows, opts)]


@pytest.mark.parametrize("V", [8195, 128256])
def test_pick_where_candidates_are_ruled_out_or_have_no_mass(V):
    """Rows whose allowed candidates are flat, few or one beside -inf, and rows so steep that a top-k cut falls among candidates whose
    mass is nothing."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    rng = np.random.default_rng(V + 1)
    rows, opts = [], []
    for kind in ("flat", "few", "one", "two", "steep", "steeper"):
        for top_k, top_p, min_p in ((0, 1.0, 0.0), (1, 1.0, 0.0), (3, 1.0, 0.0), (40, 1.0, 0.0), (40, 0.95, 0.05), (200, 0.9, 0.0),
                                    (3000, 1.0, 0.0), (0, 0.95, 0.0), (0, 1.0, 0.05), (0, 1.0, 1.0)):
            row = np.full(V, -np.inf, dtype=np.float32)
            if kind == "flat":
                allowed = rng.random(V) < 0.67
                row[allowed] = rng.standard_normal(int(allowed.sum())).astype(np.float32) * 0.05
            elif kind.startswith("steep"):      # the second best 8 and 30 below the best; everything but some forty past the span
                row[:] = rng.standard_normal(V) * 0.5 - 40.0
                row[rng.choice(V, 40, replace=False)] = rng.standard_normal(40) if kind == "steep" else -22.0
                row[V // 2] = 8.0
            else:
                n = {"few": 20, "one": 1, "two": 2}[kind]
                row[rng.choice(V, n, replace=False)] = rng.standard_normal(n)
            rows.append(row)
            draw = float(rng.integers(0, 1 << 24)) / (1 << 24)
            opts.append((float(rng.choice([0.3, 0.8, 1.3])), draw, top_k, float(np.float32(top_p)), float(np.float32(min_p))))
    f = lambda i: torch.tensor([o[i] for o in opts], dtype=torch.float32, device=dev)
    top_k = torch.tensor([o[2] for o in opts], dtype=torch.int32, device=dev)
    logits = torch.tensor(np.stack(rows), device=dev)
    want = [pick(r, *o) for r, o in zip(rows, opts)]
    got = ops.sample(logits, f(0), f(1), top_k=top_k, top_p=f(3), min_p=f(4)).cpu().tolist()
    assert [(i, g) for i, g in enumerate(got) if g != want[i]] == [(i, w) for i, w in enumerate(want) if w != got[i]], opts
    plain = ops.sample(logits, f(0), f(1)).cpu().tolist()
    assert plain == [pick(r, o[0], o[1], 0, 1.0, 0.0) for r, o in zip(rows, opts)]


def test_penalty_of_a_window_with_repeats():
    """Each occurrence of a token counts, whichever workgroup holds the token; exempt ones are left alone."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    rng = np.random.default_rng(3)
    V, W = 20000, 5
    rows = (rng.standard_normal((W, V)) * 3).astype(np.float32)
    recent = rng.integers(0, V, (W, 256)).astype(np.int32)
    recent[:, 100:180] = recent[:, 50:130]
    recent[:, 200] = -1
    recent[:, 201] = V
    n = np.array([256, 0, 1, 180, 300], dtype=np.int32)
    rp = np.array([1.1, 1.3, 2.0, 1.0, 0.7], dtype=np.float32)
    exempt = [int(recent[0, 7])]
    want = rows.copy()
    for r in range(W):
        for t in recent[r, :n[r]]:
            if 0 <= t < V and t not in exempt and rp[r] != 1.0:
                want[r, t] = want[r, t] / rp[r] if want[r, t] > 0 else want[r, t] * rp[r]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    f32 = lambda x: torch.tensor(x, dtype=torch.float32, device=dev)
    logits = f32(rows)
    ops.sample(logits, f32(np.ones(W)), f32(np.full(W, 0.5)), top_k=i32(np.zeros(W)), top_p=f32(np.ones(W)), min_p=f32(np.zeros(W)),
               repeat_penalty=f32(rp), recent=i32(recent), n_recent=i32(n), exempt=i32(exempt))
    assert np.array_equal(logits.cpu().numpy(), want)


# candidates of the bin that a cut gathers: either side of what is sorted by counting (5 to 256 keys, 64, 128 and 256 of them at a time),
# and of the network's sizes
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 65, 128, 129, 256, 257, 511, 512, 513, 1000])
def test_pick_within_a_bin_of_so_many(n):
    """One candidate far above the others, which lie in a bin or two: n in the bin that is gathered, in any order of ids."""
    import torch
    from xyntetik_runner_amd.csrc.ops import load_ops
    ops, dev = load_ops(), torch.device("cuda:0")
    rng = np.random.default_rng(n)
    V, rows, opts = 8192, [], []
    for i in range(12):
        row = np.full(V, -np.inf, dtype=np.float32)
        at = rng.permutation(V)[:n + 2]
        row[at[0]], row[at[1]] = 0.5, -20.0                     # (the row's span: bins of 0.01)
        row[at[2:]] = -0.004 - 0.004 * rng.random(n)            # (distances 0.504 to 0.508 of z: one bin)
        rows.append(row)
        opts.append((1.0, float(rng.integers(0, 1 << 24)) / (1 << 24), 0, float(np.float32(rng.choice([0.4, 0.7, 0.95, 1.0]))), 0.0))
    f = lambda i: torch.tensor([o[i] for o in opts], dtype=torch.float32, device=dev)
    top_k = torch.zeros((len(opts),), dtype=torch.int32, device=dev)
    got = ops.sample(torch.tensor(np.stack(rows), device=dev), f(0), f(1), top_k=top_k, top_p=f(3), min_p=f(4)).cpu().tolist()
    assert got == [pick(r, *o) for r, o in zip(rows, opts)]
