"""Prompts stored while a graph is being captured: nothing kept from other stores serves them."""
from __future__ import annotations

import torch

from cache_host import HostCacheModule
from test_layout_memo import BANDS, I4, I8, F16
from triattention_amd.kernels import decode as D
from triattention_amd.kernels.decode import DecodeCache


def store(cache, prompt, exact=()):
    tiles, hk = (prompt + 63) // 64, 2
    rec = lambda words: torch.zeros(hk * tiles * words, dtype=torch.int32).view(torch.uint32)
    scales, stat = torch.ones(hk * tiles * 4), torch.zeros(1, hk, 3, 128)
    kx = torch.zeros(max(1, len(exact)) * tiles * 16384, dtype=torch.uint8)
    cache.store(0, prompt, rec(2048), scales, stat, stat.clone(), {F16: None, I8: rec(2048), I4: rec(1024)},
                cache.codes(tiles)[0], BANDS, rec(1024), scales.clone(), exact, *((kx, kx.clone()) if exact else ()))
    return cache.layers[0]


def test_a_captured_store_does_not_take_a_kept_layout(monkeypatch):
    """Its bounds and task items would be uploaded, which a capture refuses: also after a store of its shape."""
    cache = DecodeCache(HostCacheModule(), max_tail=8)
    kept = store(cache, 200)["layout"]
    monkeypatch.setattr(D, "_capturing", lambda device: True)
    assert store(cache, 200)["layout"] is not kept
    assert list(cache.layouts.values()) == [kept]
    monkeypatch.setattr(D, "_capturing", lambda device: False)
    assert store(cache, 200)["layout"] is kept
