"""The draws of a batch's generators side by side against one after the other."""
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
