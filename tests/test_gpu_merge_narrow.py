"""GPU parity of the merge on narrow grids (eight waves per (sequence, q-head)).

Against the oracle's decode at the merge's own edges: split counts around one round (8 waves), the up-front loads
(16, 32, 64 splits) and past them, and tails around the score rounds (64 tokens), the value rounds (32) and their
batches.  Bar: 2e-3 max-abs and 1e-3 mean-abs, as every decode check (the partials agree to fp32 rounding).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from helpers import MAX_ABS, MEAN_ABS, bands_fn_of
from triattention_amd import synthetic as S
from triattention_amd.kernels.decode import DecodeCache
from triattention_amd.kernels.prefill import Prefill
from triattention_amd.synthetic import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles, per, tail", [(1, 1, 1), (7, 1, 31), (9, 1, 33), (17, 1, 64), (33, 1, 65), (64, 1, 127),
                                             (65, 1, 129), (70, 1, 193), (12, 5, 321)])
def test_narrow_merge_matches_the_oracle(module, tiles, per, tail):
    print(f"\n[merge] {tiles} tiles in runs of {per}, tail {tail}", flush=True)
    hq, hk, prompt, scale = 6, 2, 64 * tiles - 3, 128 ** -0.5
    g = S.gen(9000 + tiles)
    k, v = S.outlier_tensor(g, 1, hk, prompt), S.outlier_tensor(g, 1, hk, prompt)
    bands = torch.tensor([[S.INF, S.INF]] * 3 + [[1, S.INF]] * 3, dtype=torch.int32)
    cache = DecodeCache(module, max_tail=tail)
    cache.per, cache.out_dtype = per, torch.float32
    assert hq < cache.SHORT_WIDE * module.device_cus()
    pre = Prefill(module, bands_fn_of(bands), cache)
    pre.store_only(0, k.cuda(), v.cuda(), hq)
    kt, vt = S.outlier_tensor(g, tail, hk, 1)[:, :, 0], S.outlier_tensor(g, tail, hk, 1)[:, :, 0]
    q = S.outlier_tensor(g, 1, hq, 1)
    for name, rows in (("tail_k", kt), ("tail_v", vt)):
        cache.layers[0][name][0, :, :tail - 1] = rows[:tail - 1].transpose(0, 1).cuda()
    cache.step.fill_(tail - 1)
    cache.host_step = tail - 1
    out = cache(0, q.cuda(), kt[-1][None, :, None].cuda().contiguous(), vt[-1][None, :, None].cuda().contiguous(), scale)
    codes = O.prefill_codes(None, bits(k[0]), bits(v[0]), bands.numpy(), decode_cache=True)
    tk, tv = (np.ascontiguousarray(bits(x.transpose(0, 1).contiguous())) for x in (kt, vt))
    ref = O.decode(codes, bands.numpy(), bits(q[0, :, 0]), prompt, cache.split_of(0, 0), scale, tk, tv,
                   bits(kt[-1].contiguous()), bits(vt[-1].contiguous()), tail - 1)
    err = np.abs(out[0, :, 0].cpu().numpy() - ref)
    assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS, f"max {err.max():.3e} mean {err.mean():.3e}"
