"""The draws of a batch's generators side by side against one after the other."""
import struct

import numpy as np
import pytest


@pytest.mark.parametrize("n", [1, 7, 8, 64])
@pytest.mark.parametrize("every", [0, 2, 5])
def test_draws_side_by_side(n, every):
    from xyntetik_runner_amd.sampling.params import SamplerState, SamplingParams, draws
    mk = lambda: [SamplerState(SamplingParams(temperature=0.0 if every and i % every == 0 else 0.8, seed=(i << 57) + i * 977 + 1)) for i in range(n)]
    many, one = mk(), mk()
    greedy = [s.params.greedy for s in many]
    for _ in range(20):
        assert draws(many, greedy) == [0.0 if s.params.greedy else s.draw() for s in one]
    assert [s.rng for s in many] == [s.rng for s in one] and all(type(s.rng) is int for s in many)
    twice = [many[0]] * 9
    assert draws(twice, [greedy[0]] * 9) == [0.0 if greedy[0] else one[0].draw() for _ in range(9)]


@pytest.mark.parametrize("top_k,kept", [(40, 40), (40.0, 40), (40.7, 40), (0.5, 0), (True, 1), (np.float32(7), 7), (np.int64(9), 9), (1e12, 0x7FFFFFFF),
                                        (float("inf"), 0x7FFFFFFF), (float("nan"), 0)])
def test_top_k_of_any_number(top_k, kept):
    """Options are numbers of any type, as they come from a request's JSON: the kernels get the whole part (no number: no cut)."""
    from xyntetik_runner_amd.sampling.params import SamplerState, SamplingParams
    for temperature in (0.8, 1e39):         # (the latter is beyond 32 bits)
        words = SamplerState(SamplingParams(temperature=temperature, top_k=top_k, top_p=0.5)).words
        assert struct.unpack("=4fi", words)[1:] == (0.5, 0.0, 1.0, kept)


@pytest.mark.parametrize("n", [1, 8, 64])
@pytest.mark.parametrize("every", [0, 3])
def test_draws_as_the_kernels_get_them(n, every):
    """What a batch stores into its options: the same 32-bit numbers, whether they come as a list or side by side."""
    from xyntetik_runner_amd.sampling.params import SamplerState, SamplingParams, draw_values
    mk = lambda: [SamplerState(SamplingParams(temperature=0.0 if every and i % every == 0 else 0.8, seed=i * 977 + 5)) for i in range(n)]
    many, one = mk(), mk()
    stored = np.empty(n, dtype=np.float32)
    for _ in range(3):
        stored[:] = draw_values(many, [s.greedy for s in many])
        assert stored.tolist() == [0.0 if s.greedy else s.draw() for s in one]
