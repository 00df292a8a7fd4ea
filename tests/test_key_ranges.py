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


@pytest.mark.parametrize("B,heads", [(1, 1), (1, 2), (1, 8), (1, 100), (4, 1), (8, 1), (8, 8), (16, 8), (32, 8), (64, 8), (512, 32)])
@pytest.mark.parametrize("table_tiles", [7, 16, 64, 640, 5000])
def test_longest_request_of_a_key(B, heads, table_tiles):
    """What a graph keeps room for is what the longest request with its key would ask for, whatever it is recorded with."""
    from xyntetik_runner_amd.engine.graphs import most_tiles
    of = {}
    for tiles in range(1, table_tiles + 1):
        of.setdefault(splits_for(B, tiles, heads), []).append(tiles)
    for ranges, tiles in of.items():
        assert most_tiles(B, ranges, heads, table_tiles) == tiles[-1], (ranges, tiles[0], tiles[-1])


@pytest.mark.gpu
def test_results_do_not_hang_on_the_length_that_was_recorded(tmp_path):
    """A request of 900 keys on the graph that one of 520 had recorded, and on its own: the same key ranges, so the same bits."""
    from tiny import make_model, prompt_ids
    from xyntetik_runner_amd.engine.batch import StepEntry
    from xyntetik_runner_amd.engine.runner import ModelRunner
    d = make_model("D", str(tmp_path))
    toks = {n: prompt_ids(n + 3, 1000, n) for n in (520, 900)}

    def decoded(lens):
        runner = ModelRunner.from_folder(d, dtype="bfloat16", max_tokens=2048, page_size=64, max_requests=2)
        for i, n in enumerate(lens):
            runner.step([StepEntry(i, toks[n][:n], [])])
            rows = [runner.step([StepEntry(i, [t], [0])]).cpu().numpy() for t in toks[n][n:]]
        assert runner.graphs.captures == 1
        (ctx, _, _), = runner.graphs.graphs.values()
        return [p.n_few for p in ctx._plans.values()], np.stack(rows)

    after, alone = decoded([520, 900]), decoded([900])
    assert after[0] == alone[0] and min(alone[0]) >= 8
    assert np.array_equal(after[1], alone[1])


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
