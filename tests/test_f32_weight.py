"""A 32-bit weight that a model keeps takes every way of a plain matrix: copies, files, parameters."""
import copy
import io
import pickle

import torch

from xyntetik_runner_amd.csrc.ops import F32Weight


def test_copies_files_and_parameters():
    w = torch.randn(6, 512).as_subclass(F32Weight)
    twice = copy.deepcopy({"a": [w, torch.zeros(1)], "b": w, "rows": w.as_subclass(torch.Tensor)[2:4]})
    new = twice["a"][0]
    assert isinstance(new, F32Weight) and new is twice["b"] and torch.equal(new, w) and new.data_ptr() != w.data_ptr()
    assert twice["rows"].data_ptr() == new.data_ptr() + 2 * 512 * 4 and twice["a"][1].shape == (1,)    # one memory, as before
    assert isinstance(copy.copy(w), F32Weight)
    f = io.BytesIO()
    torch.save({"w": w}, f)
    f.seek(0)
    for read in (torch.load(f, weights_only=True)["w"], pickle.loads(pickle.dumps(w))):
        assert type(read) is torch.Tensor and torch.equal(read, w)
    p = torch.nn.Parameter(w, requires_grad=False)
    assert isinstance(p, torch.nn.Parameter) and p.data_ptr() == w.data_ptr()
    assert all(type(x) is torch.Tensor for x in (w[:2], w + 1, w.t(), torch.cat([w, w]), w.clone()))
