"""A decode step's kept plan: by the values and shapes of the call, never by an argument's identity."""
from __future__ import annotations

import types

import numpy as np
import pytest
import torch

from cache_host import HostCacheModule
from test_layout_memo import store
from triattention_amd.kernels.decode import DecodeCache


class Module(HostCacheModule):
    """Records the scale that each step's launch applies."""

    def __init__(self):
        self.scales, self.plans = [], 0

    def plan_decode(self, *args, **kw):
        self.plans += 1
        step = lambda *a, **k: self.scales.append(args[25])
        return types.SimpleNamespace(run=step, launch=step)


@pytest.mark.parametrize("kind", [np.array, torch.tensor])
def test_a_scale_changed_in_place_is_applied(kind):
    module = Module()
    cache = DecodeCache(module, max_tail=8)
    store(cache, 0, 200)
    q, k, v = (torch.zeros(1, h, 1, 128, dtype=torch.bfloat16) for h in (4, 2, 2))
    scale = kind(0.125)
    for value in (0.125, 0.5, 0.5, 0.125):
        scale[...] = value
        cache(0, q, k, v, scale)
    assert module.scales == [0.125, 0.5, 0.5, 0.125]
    # new objects of one value share the plan
    for _ in range(3):
        cache(0, q, k, v, kind(0.5))
    assert module.plans == 2 and len(cache.layers[0]["calls"]) == 2
