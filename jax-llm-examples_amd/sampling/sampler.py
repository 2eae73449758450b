"""Chooses next tokens from float32 logits on the device, one kernel call per step."""
from __future__ import annotations

from typing import Sequence

import torch

from .params import SamplingParams


class Sampler:
    def __init__(self, ops, device) -> None:
        self.ops = ops
        self.device = torch.device(device)

    def __call__(self, logits: torch.Tensor, params: Sequence[SamplingParams], counters: Sequence[int]) -> list[int]:
        """``counters[i]``: how many tokens request ``i`` has generated so far (it numbers
        the random draw, so a request's draws do not depend on the batch)."""
        m = logits.shape[0]
        assert m == len(params) == len(counters)
        topk, seeds = [int(p.sample_topk) for p in params], [int(p.seed) & 0x7FFFFFFF for p in params]
        ctr = [int(c) & 0x7FFFFFFF for c in counters]
        if hasattr(self.ops, "greedy") and all(p.greedy for p in params) and all(-2 ** 31 <= k < 2 ** 31 for k in topk):
            return self.ops.greedy(logits)[0]  # (nothing to bring to the device first)
        temp = torch.tensor([0.0 if p.greedy else float(p.sample_temp) for p in params], dtype=torch.float32)
        dev = self.device
        packed = torch.tensor([topk, seeds, ctr], dtype=torch.int32).to(dev)  # one copy for the three integer rows
        any_top_k = any(not p.greedy and 0 < p.sample_topk for p in params)
        out = self.ops.sample(logits, temp.to(dev), packed[0], packed[1], packed[2], any_top_k=any_top_k)
        return [int(t) for t in out.cpu().tolist()]

    def greedy(self, logits: torch.Tensor):
        """The largest logit of each row, lowest id among equals, and a copy of the logits."""
        if hasattr(self.ops, "greedy"):
            return self.ops.greedy(logits, copy=True)
        m = logits.shape[0]
        return self(logits, [SamplingParams()] * m, [0] * m), logits.clone()
