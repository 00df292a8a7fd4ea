"""Picking the next token of every row of a step on the device.

One kernel call takes all rows: greedy rows and sampled rows together.  The host
supplies each sampled row's draw from its request's generator, so a request's tokens
depend on its own seed only, not on what else is in the batch.
"""
from __future__ import annotations

from typing import List, Optional, Sequence

import numpy as np
import torch

from .params import RECENT_WINDOW, SamplerState, draws


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
        params = [s.params for s in states]
        temps = [p.temperature for p in params]
        greedy = [not (t > 0.0) for t in temps]
        penalties = [p.repeat_penalty for p in params]
        # floats: temp, top_p, min_p, rp, draw ; ints: top_k, n_recent ; window
        need_window = any(x != 1.0 and not g for x, g in zip(penalties, greedy))
        nf = 5 * W
        ni = 2 * W + (W * RECENT_WINDOW if need_window else 0)
        host = torch.empty((nf + ni,), dtype=torch.int32, pin_memory=True)
        h = host.numpy()
        hf, hi = h[:nf].view(np.float32).reshape(5, W), h[nf:]
        hf[0] = temps if not any(greedy) else [0.0 if g else t for t, g in zip(temps, greedy)]
        hf[1] = [p.top_p for p in params]
        hf[2] = [p.min_p for p in params]
        hf[3] = penalties
        hf[4] = draws(states, greedy)
        hi[:W] = [p.top_k for p in params]
        hi[W:2 * W] = [s.n_recent for s in states]
        if need_window:
            win = hi[2 * W:].reshape(W, RECENT_WINDOW)
            for r, s in enumerate(states):
                win[r, :] = s.recent
        dev = host.to(self.device, non_blocking=True)
        if all(greedy):
            temp, _, _, _, draw = dev[:nf].view(torch.float32).view(5, W).unbind(0)
            return self.ops.sample(logits, temp, draw)
        return self.ops.sample_packed(logits, dev, RECENT_WINDOW if need_window else 0, exempt=self.exempt)
