"""Picking the next token of every row of a step on the device.

One kernel call takes all rows: greedy rows and sampled rows together.  The host
supplies each sampled row's draw from its request's generator, so a request's tokens
depend on its own seed only, not on what else is in the batch.
"""
from __future__ import annotations

from array import array
from typing import List, Optional, Sequence

import numpy as np
import torch

from .params import RECENT_WINDOW, SamplerState, draw_values


class Sampler:
    def __init__(self, ops, device, exempt_ids: Sequence[int] = ()):
        self.ops, self.device = ops, device
        ex = [int(t) for t in exempt_ids]          # (the kernel walks the list, however long)
        self.exempt = torch.tensor(ex, dtype=torch.int32, device=device) if ex else None

    @staticmethod
    def uses_history(states: List[SamplerState]) -> bool:
        """Whether a row's pick depends on the tokens its request got before (a repeat penalty)."""
        return any((not s.params.greedy) and s.params.repeat_penalty != 1.0 for s in states)

    def sample(self, logits: torch.Tensor, states: List[SamplerState]) -> List[int]:
        """``logits [W, V]`` float32 on the device, one state per row -> token ids."""
        if logits.shape[0] == 0:
            return []
        return [int(t) for t in self.launch(logits, states).cpu().tolist()]

    def launch(self, logits: torch.Tensor, states: List[SamplerState]) -> torch.Tensor:
        """The same without waiting for the result: token ids ``[W]`` int32 on the device."""
        W = logits.shape[0]
        assert W == len(states) and W > 0
        greedy = [s.greedy for s in states]
        # floats: temp, top_p, min_p, rp, draw ; ints: top_k, n_recent ; window.  (Every state keeps its options as words: a batch of 64 is
        # one join and one transposed copy, 25 us less than a list and its conversion an option, and 64 windows 6 us instead of 200.)
        need_window = any([s.penalised for s in states])
        nf = 5 * W
        ni = 2 * W + (W * RECENT_WINDOW if need_window else 0)
        host = torch.empty((nf + ni,), dtype=torch.int32, pin_memory=True)
        h = host.numpy()
        options = h[:7 * W].reshape(7, W)
        words = np.frombuffer(b"".join([s.words for s in states]), dtype=np.int32).reshape(W, 5).T
        options[:4], options[5] = words[:4], words[4]
        options[4].view(np.float32)[:] = draw_values(states, greedy)
        options[6] = [s.n_recent for s in states] if need_window else 0
        if need_window:
            h[7 * W:] = np.frombuffer(b"".join([s.recent if type(s.recent) is array else array("i", s.recent) for s in states]), dtype=np.int32)
        dev = host.to(self.device, non_blocking=True)
        if all(greedy):
            temp, _, _, _, draw = dev[:nf].view(torch.float32).view(5, W).unbind(0)
            return self.ops.sample(logits, temp, draw)
        return self.ops.sample_packed(logits, dev, RECENT_WINDOW if need_window else 0, exempt=self.exempt)
