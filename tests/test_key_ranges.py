"""Into how many ranges of keys a recorded decode step cuts its requests, on either side of what changes it."""
import numpy as np
import pytest

from xyntetik_runner_amd.engine.graphs import splits_for


# (requests, tiles of 32 keys, key/value heads): one range up to 15 tiles from 8 workgroups on; fewer workgroups, and 16 tiles and more, as many
# ranges of 4 tiles or longer as make one round of 256 workgroups, a power of two of them
@pytest.mark.parametrize("args,ranges", [((1, 15, 8), 1), ((1, 16, 8), 4), ((4, 15, 2), 1), ((4, 16, 2), 4), ((8, 15, 1), 1), ((8, 16, 1), 4),
                                         ((1, 15, 7), 2), ((1, 16, 7), 4), ((1, 15, 1), 2), ((1, 8, 2), 2), ((1, 7, 2), 1), ((1, 1, 1), 1),
                                         ((1, 32, 8), 8), ((1, 1000, 8), 32), ((16, 1000, 8), 2), ((64, 15, 8), 1), ((64, 1000, 8), 1)])
def test_splits_for(args, ranges):
    assert splits_for(*args) == ranges


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_decoding_from_one_range_into_several(tmp_path, dtype):
    """Four requests of two key/value heads, the longest from 470 keys to 500: recorded with one range a request, then with four."""
    import plain_llama as P
    from test_replay_gpu import TOL
    from tiny import logit_error, make_model, prompt_ids
    from xyntetik_runner_amd.engine.batch import StepEntry
    from xyntetik_runner_amd.engine.runner import ModelRunner
    d = make_model("A", str(tmp_path))
    cfg, w = P.load_folder(d)
    lens, n_dec = [470, 300, 33, 1], 30
    toks = [prompt_ids(n + n_dec, cfg["vocab_size"], 900 + i) for i, n in enumerate(lens)]
    runner = ModelRunner.from_folder(d, dtype=dtype, max_tokens=1024, page_size=16, max_requests=4)
    runner.step([StepEntry(i, t[:n], []) for i, (t, n) in enumerate(zip(toks, lens))])
    got = []
    for k in range(n_dec):
        got.append(runner.step([StepEntry(i, [t[n + k]], [0]) for i, (t, n) in enumerate(zip(toks, lens))]).cpu().numpy())
    # (481 keys are 16 tiles: the longest request's twelfth token)
    assert sorted(key[1] for key in runner.graphs.graphs) == [1, 4] and runner.graphs.captures == 2 and runner.graphs.replays == n_dec - 2
    for i, (t, n) in enumerate(zip(toks, lens)):
        want = P.forward(cfg, w, t)[n:]
        rows = np.stack([g[i] for g in got])
        for part in (slice(0, 11), slice(11, None)):
            mx, mean = logit_error(rows[part], want[part])
            assert mx <= TOL[dtype][0] and mean <= TOL[dtype][1], (i, part, mx, mean)
