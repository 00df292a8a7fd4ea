"""Which portions of a step run retention and the delta rule in chunks (a division of the step's requests, made on the host)."""
import pytest

from xyntetik_runner_amd.csrc.ops import Ops


@pytest.fixture
def ops():
    return Ops.__new__(Ops)         # (no library and no device: the division is arithmetic)


@pytest.mark.parametrize("kind", ["delta", "retention"])
@pytest.mark.parametrize("H", [16, 32])
def test_division_of_a_step(ops, kind, H):
    rows = lambda *q_lens: ops.chunked_rows(kind, q_lens, H, 128)
    # decoded tokens and short portions never, a long portion always, also beside decoded tokens, which stay out of it
    assert rows(*[1] * 64) is None and rows(95) is None
    assert rows(128) == 128 and rows(2048) == 2048 and rows(1, 1, 400, *[1] * 61) == 400
    assert rows(1, 2048, *[1] * 62) == 2048
    # many portions of one length fill the chip row by row, and chunks would only pad them
    assert rows(*[100] * 20) is None


def test_scratch_is_bounded(ops, monkeypatch):
    monkeypatch.setattr(Ops, "CHUNKS_SCRATCH", 10 * Ops._chunk_floats("delta", 32))
    assert ops.chunked_rows("delta", [640], 32, 128) == 640 and ops.chunked_rows("delta", [641], 32, 128) is None


# a workgroup a (request, head): on either side of how many of them are still the faster way, by the values' size
@pytest.mark.parametrize("kind,Dv,most", [("retention", 16, 1024), ("delta", 16, 1024), ("retention", 17, 2048), ("delta", 17, 4096), ("retention", 64, 2048),
                                          ("delta", 64, 4096), ("retention", 65, None), ("delta", 128, None)])
def test_where_a_step_in_one_kernel_pays(kind, Dv, most):
    from types import SimpleNamespace
    from xyntetik_runner_amd.csrc.ops import Ops
    pays = lambda B, H, **kw: Ops.recurrence_step_pays(kind, SimpleNamespace(max_q_len=kw.get("rows", 1), B=B), B, H, kw.get("D", 64), Dv)
    assert pays(1, 1) and pays(8, 32) and not pays(8, 32, rows=2) and not pays(8, 32, D=32)
    if most is None:
        assert pays(512, 64)
    else:
        assert pays(most // 32, 32) and not pays(most // 32 + 1, 32)
