"""Decode of caches with exact heads from the task table against the gather from the metadata rows.

The two launches read the same entries, so every output is equal bit for bit: uniform and balanced splits,
one exact head and all of them, ragged batches, groups in both lane layouts."""
from __future__ import annotations

import pytest
import torch

from helpers import bands_fn_of
from triattention_amd import synthetic as S
from triattention_amd.kernels.decode import DecodeCache
from triattention_amd.kernels.prefill import Prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq, hk, exact, prompts, per", [
    (6, 2, [1], (64,), None), (6, 2, [0, 1], (65, 1, 700), None), (14, 2, [0], (1100, 130), None),
    (14, 2, [1], (1100, 130), 3), (8, 8, [2, 5], (333,), 2), (4, 1, [0], (2000,), None)])
def test_task_table_equals_the_gather(module, hq, hk, exact, prompts, per):
    g = S.gen(9500 + hq + hk)
    group = hq // hk
    bands = torch.tensor([[S.INF, S.INF] if r % 2 else [1 + r % 5, S.INF] for r in range(hk) for _ in range(group)],
                         dtype=torch.int32)
    kv = [(S.outlier_tensor(g, 1, hk, n).cuda(), S.outlier_tensor(g, 1, hk, n).cuda()) for n in prompts]
    q, k, v = (S.outlier_tensor(g, len(prompts), h, 1).cuda() for h in (hq, hk, hk))
    outs = []
    for tasks in (True, False):
        cache = DecodeCache(module, max_tail=4)
        cache.ragged, cache.tasks, cache.per, cache.out_dtype = True, tasks, per, torch.float32
        pre = Prefill(module, bands_fn_of(bands, exact), cache)
        for pk, pv in kv:
            pre.store_only(0, pk, pv, hq)
        outs.append(cache(0, q, k, v, 128 ** -0.5).clone())
        assert ("tasks" in cache.layers[0]) == tasks
    assert torch.equal(*outs)


def test_a_table_is_ignored_with_exact_heads_unless_it_says_that_it_lists_them(module, monkeypatch):
    """n_tasks > 0 with xslot gathers: a table of one split and partials never cleared change nothing."""
    g = S.gen(9600)
    cache = DecodeCache(module, max_tail=4)
    cache.out_dtype = torch.float32
    bands = torch.tensor([[S.INF, S.INF]] * 3 + [[1, S.INF]] * 3, dtype=torch.int32)
    pk, pv = (S.outlier_tensor(g, 1, 2, 900).cuda() for _ in range(2))
    Prefill(module, bands_fn_of(bands, [1]), cache).store_only(0, pk, pv, 6)
    calls = []
    real = module.plan_decode
    monkeypatch.setattr(module, "plan_decode", lambda *a, **kw: calls.append((a, kw)) or real(*a, **kw))
    q, k, v = (S.outlier_tensor(g, 1, h, 1).cuda() for h in (6, 2, 2))
    cache(0, q, k, v, 128 ** -0.5)
    args, kw = calls[-1]
    args = list(args)
    table, n = args[30]
    assert kw["exact_tasks"] and n > 1
    outs = []
    for tasks, exact_tasks in (((table, n), True), ((table[:512], 1), False)):
        if not exact_tasks:
            args[20:23] = [torch.full_like(x, 7.0) for x in args[20:23]]
        args[19] = torch.empty_like(args[19])
        args[30], kw["exact_tasks"] = tasks, exact_tasks
        real(*args, **kw).run(q, k, v, args[19])
        outs.append(args[19])
    assert torch.equal(*outs)
