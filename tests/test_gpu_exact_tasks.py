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
