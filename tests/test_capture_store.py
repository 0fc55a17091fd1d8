"""Prompts stored while a graph is being captured: nothing kept from other stores serves them, and nothing read
from the first replay's prompt serves the next one's."""
from __future__ import annotations

import types

import pytest
import torch

from cache_host import HostCacheModule
from test_layout_memo import BANDS, I4, I8, F16
from triattention_amd.kernels import decode as D
from triattention_amd.kernels.decode import DecodeCache


class Module(HostCacheModule):
    """Records the task table that each planned step reads."""

    def __init__(self):
        self.tables, self.built = [], 0

    def decode_tasks(self, *args):
        self.built += 1
        return object(), 1

    def plan_decode(self, *args, **kw):
        self.tables.append(args[-1])
        step = lambda *a, **k: None
        return types.SimpleNamespace(run=step, launch=step)


def store(cache, prompt, exact=()):
    tiles, hk = (prompt + 63) // 64, 2
    rec = lambda words: torch.zeros(hk * tiles * words, dtype=torch.int32).view(torch.uint32)
    scales, stat = torch.ones(hk * tiles * 4), torch.zeros(1, hk, 3, 128)
    kx = torch.zeros(max(1, len(exact)) * tiles * 16384, dtype=torch.uint8)
    cache.store(0, prompt, rec(2048), scales, stat, stat.clone(), {F16: None, I8: rec(2048), I4: rec(1024)},
                cache.codes(tiles)[0], BANDS, rec(1024), scales.clone(), exact, *((kx, kx.clone()) if exact else ()))
    return cache.layers[0]


def step(cache):
    q, k, v = (torch.zeros(1, h, 1, 128, dtype=torch.bfloat16) for h in (4, 2, 2))
    cache(0, q, k, v, 0.1)


def test_a_captured_store_does_not_take_a_kept_layout(monkeypatch):
    """Its bounds and task items would be uploaded, which a capture refuses: also after a store of its shape."""
    cache = DecodeCache(Module(), max_tail=8)
    kept = store(cache, 200)["layout"]
    monkeypatch.setattr(D, "_capturing", lambda device: True)
    assert store(cache, 200)["layout"] is not kept
    assert list(cache.layouts.values()) == [kept]
    monkeypatch.setattr(D, "_capturing", lambda device: False)
    assert store(cache, 200)["layout"] is kept


@pytest.mark.parametrize("exact", [(), (1,)])
def test_steps_after_a_captured_store_read_no_table(monkeypatch, exact):
    """A table holds the K scales of the prompt that was there when it was built."""
    cache = DecodeCache(Module(), max_tail=8)
    cache.per = 2  # (uniform runs: nothing to upload)
    monkeypatch.setattr(D, "_capturing", lambda device: True)
    store(cache, 200, exact)
    monkeypatch.setattr(D, "_capturing", lambda device: False)
    step(cache)
    assert cache.module.tables == [None] and cache.module.built == 0
    store(cache, 200, exact)  # (an eager store has its table again)
    step(cache)
    assert cache.module.tables[1] is not None and cache.module.built == 1
