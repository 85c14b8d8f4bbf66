"""Workspace buffer cache, as local_experiments/video_runtime_v1/attention.py:7-13.

Buffers are keyed by (name, shape, device, dtype) and reused across calls, so a
returned output tensor is overwritten by the next call with the same key.
"""
from __future__ import annotations

import torch


class Workspace:
    def __init__(self):
        self.entries = {}

    def tensor(self, name, shape, device, dtype):
        # torch.Size is a tuple: equal shapes are equal keys in either form
        key = (name, shape if isinstance(shape, tuple) else tuple(shape),
               device if isinstance(device, torch.device) else torch.device(device), dtype)
        buf = self.entries.get(key)
        if buf is None:
            buf = self.entries[key] = torch.empty(shape, device=device, dtype=dtype)
        return buf

    def bytes(self):
        return sum(x.numel() * x.element_size() for x in self.entries.values())
