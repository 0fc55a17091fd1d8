"""The decode cache's shared split layouts: by shape and bands, bounded, and equal to a fresh computation."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from cache_host import HostCacheModule
from triattention_amd.kernels.decode import DecodeCache, balanced_partition, entry_costs, sequence_metadata, \
    split_bounds
from triattention_amd.kernels.prefill import F16, I4, I8
from triattention_amd.synthetic import INF

BANDS = torch.tensor([[INF, INF], [1, INF], [2, 4], [1, 1]], dtype=torch.int32)


def store(cache, layer, prompt, batch=1, bands=BANDS, value=1.0, hk=2):
    tiles = (prompt + 63) // 64
    n = batch * hk * tiles
    rec = lambda words: torch.full((n * words,), int(value), dtype=torch.int32).view(torch.uint32)
    scales = torch.full((n * 4,), value)
    stat = torch.full((batch, hk, 3, 128), value)
    cache.store(layer, prompt, rec(2048), scales, stat, stat.clone(), {F16: None, I8: rec(2048), I4: rec(1024)},
                cache.codes(tiles)[0], bands, rec(1024), scales.clone())
    return cache.layers[layer]


def test_prompts_of_one_shape_share_a_layout_and_keep_their_own_data():
    cache = DecodeCache(HostCacheModule(), max_tail=8)
    a, b = store(cache, 0, 200, value=1.0), store(cache, 1, 200, value=2.0)
    assert a["layout"] is b["layout"] and len(cache.layouts) == 1
    assert a["ka"].data_ptr() != b["ka"].data_ptr()
    assert bool((a["ka"] == 1).all()) and bool((b["ka"] == 2).all())
    for e in (a, b):
        assert not e["tail_k"].any() and not e["tail_v"].any() and e["store"].arrays["tail_base"].tolist() == [0, 0]
    # the last tile's length, the batch, the bands and a forced split each give a layout of their own
    assert store(cache, 2, 200, batch=2)["layout"] is not a["layout"]
    assert store(cache, 3, 264)["layout"] is not a["layout"]
    assert store(cache, 4, 200, bands=BANDS.flip(0))["layout"] is not a["layout"]
    cache.per = 1
    assert store(cache, 5, 200)["layout"]["bounds"] is None


@pytest.mark.parametrize("prompt, batch", [(1, 1), (64, 3), (65, 1), (1100, 2), (4000, 1)])
def test_a_shared_layout_equals_a_fresh_one(prompt, batch):
    shared = DecodeCache(HostCacheModule(), max_tail=8)
    store(shared, 0, prompt, batch)
    again = store(shared, 0, prompt, batch)
    fresh = store(DecodeCache(HostCacheModule(), max_tail=8), 0, prompt, batch)
    assert again["per"] == fresh["per"] and again["splits"] == fresh["splits"]
    assert np.array_equal(again["bounds_host"], fresh["bounds_host"])
    assert np.array_equal(DecodeCache._task_items(again), DecodeCache._task_items(fresh))


def bisected(meta, batch, slots):
    """The partition by sixty steps of bisection over the target cost of a run, whatever the cache's size."""
    costs, count = entry_costs(meta), meta["count"].numpy()
    heads, floor = costs.sum(1), np.maximum((count + 63) // 64, 1)
    runs = lambda t: np.maximum(np.minimum(np.ceil(heads / t), count), floor)
    lo, hi = float(costs[costs > 0].min()), float(heads.max()) + 1
    if batch * runs(hi).sum() <= slots:
        for _ in range(60):
            mid = (lo + hi) / 2
            lo, hi = (lo, mid) if batch * runs(mid).sum() <= slots else (mid, hi)
    n = runs(hi).astype(np.int64)
    while True:
        b = split_bounds(costs, meta["valid"].numpy(), n)
        if (np.diff(b, axis=1) <= 64).all():
            return b
        n = n + (np.diff(b, axis=1) > 64).any(1)


@pytest.mark.parametrize("tiles, batch, exact", [
    (1, 1, []), (1, 5, [0]), (33, 1, [1]), (64, 1, []), (64, 4, [0, 1]), (64, 9, [0]), (256, 2, [1]), (511, 2, []),
    (2048, 1, [0]), (300, 9, [])])
@pytest.mark.parametrize("slots", [8, 1024])
def test_a_short_cache_is_cut_without_bisection(monkeypatch, tiles, batch, exact, slots):
    """A cache whose every run may be one tile is cut in one evaluation, to the bounds that bisection gives (a new
    prompt length pays for this on the host)."""
    codes = DecodeCache(HostCacheModule()).codes(tiles)[0]
    meta = sequence_metadata(BANDS, tiles, 2, codes, exact)
    want = bisected(meta, batch, slots)
    evaluations, ceil = [], np.ceil
    monkeypatch.setattr(np, "ceil", lambda x: evaluations.append(1) or ceil(x))
    (got,), splits = balanced_partition([meta], [batch], slots)
    assert splits == want.shape[1] - 1 and np.array_equal(got.numpy(), want)
    assert len(evaluations) <= (2 if batch * int(meta["count"].sum()) <= slots else 63)


@pytest.mark.parametrize("per", [None, 3])
@pytest.mark.parametrize("grow", [0, 128])
def test_task_items_are_the_kept_splits_costliest_first(per, grow):
    """Against every split's entries added up one by one, over stores of several lengths and batches."""
    cache = DecodeCache(HostCacheModule(), max_tail=64, grow_tail=grow)
    cache.ragged, cache.per = True, per
    for prompt, batch in ((200, 2), (64, 1), (1500, 1), (130, 3)):
        store(cache, 0, prompt, batch)
    e = cache.layers[0]
    costs = {}
    for g in e["groups"]:
        tile_costs, count = entry_costs(g["meta"]), g["meta"]["count"].tolist()
        for s in range(g["row0"], g["row0"] + g["batch"]):
            for h in range(2):
                for i in range(e["splits"]):
                    first, end = (i * e["per"], min((i + 1) * e["per"], count[h])) if e["bounds_host"] is None else \
                        e["bounds_host"][s, h, i:i + 2].tolist()
                    if first < end:  # (a growth split holds no kept tile yet: listed, at no cost)
                        costs[(s * 2 + h) * e["splits"] + i] = tile_costs[h, first:min(end, count[h])].sum()
    assert DecodeCache._task_items(e).tolist() == sorted(costs, key=lambda i: (-costs[i], i))


def test_layouts_are_bounded():
    cache = DecodeCache(HostCacheModule(), max_tail=8)
    cache.LAYOUTS = 3
    for tiles in range(1, 7):
        store(cache, 0, 64 * tiles)
    assert len(cache.layouts) == 3
    assert store(cache, 0, 64)["splits"] >= 1 and len(cache.layouts) == 3


def test_layouts_are_dropped_under_another_threads_feet():
    """Two stores that drop the same layout: the second finds it gone, or the dict changed while it looked."""
    class Racing(dict):
        def __iter__(self):
            for key in list(dict.__iter__(self)):
                dict.pop(self, key, None)  # the other thread's drop, between finding a key and dropping it
                yield key

    cache = DecodeCache(HostCacheModule(), max_tail=8)
    cache.LAYOUTS = 1
    store(cache, 0, 64)
    cache.layouts = Racing(cache.layouts)
    store(cache, 0, 128)


def test_growth_turned_on_later_leaves_earlier_sequences_without_room(monkeypatch):
    """tail_spill follows a row's growth regions wherever its first word is not negative."""
    # (77: what an unwritten allocation may hold)
    monkeypatch.setattr(torch, "empty", lambda shape, dtype, **kw: torch.zeros(shape, dtype=dtype).fill_(77)
                        if dtype != torch.uint32 else torch.zeros(shape, dtype=dtype))
    cache = DecodeCache(HostCacheModule(), max_tail=64)
    store(cache, 0, 200)
    cache.ragged, cache.grow_tail = True, 128
    store(cache, 0, 130)
    grow = cache.layers[0]["store"].arrays["grow"]
    assert bool((grow[0] == -1).all()) and bool((grow[1, :, 0] >= 0).all())


@pytest.mark.gpu
def test_layouts_are_shared_within_one_stream(module):
    from helpers import bands_fn_of
    from triattention_amd.kernels.prefill import Prefill

    cache = DecodeCache(module, max_tail=8)
    pre = Prefill(module, bands_fn_of(BANDS), cache)
    kv = torch.ones(1, 2, 200, 128, device="cuda", dtype=torch.bfloat16)
    q = torch.ones(1, 4, 1, 128, device="cuda", dtype=torch.bfloat16)
    other = torch.cuda.Stream()
    layouts, outs = [], []
    for stream in (None, None, other, other):
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            pre.store_only(0, kv, kv, 4)
            outs.append(cache(0, q, kv[:, :, :1].contiguous(), kv[:, :, :1].contiguous(), 0.1))
        layouts.append(cache.layers[0]["layout"])
    torch.cuda.synchronize()
    assert layouts[0] is layouts[1] and layouts[2] is layouts[3] and layouts[0] is not layouts[2]
    assert all(torch.equal(outs[0], o) for o in outs)
