"""GPU parity of the merge on narrow grids (four or eight waves per (sequence, q-head)).

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


@pytest.mark.parametrize("batch, tail, splits", [(1, 32, 64), (1, 33, 64), (1, 1, 65), (43, 1, 2), (43, 192, 3),
                                                 (43, 193, 3)])
def test_narrow_merge_around_its_choice_of_waves(module, batch, tail, splits):
    """Either side of the tails and split counts at which the wave count changes, on grids of up to and of more than
    a workgroup per CU: the merge of given partials and tail rows against the same sums in float64, each
    (sequence, q-head) of its own; and a replay gives an eager step's bits."""
    hq, hk, scale = 6, 2, 128 ** -0.5
    assert (batch * hq <= module.device_cus()) == (batch == 1) and batch * hq < 2 * module.device_cus()
    print(f"\n[merge] {batch} sequences, tail {tail}, {splits} splits", flush=True)
    g = S.gen(9200 + tail)
    prompt = 64 * splits
    k, v = (S.outlier_tensor(g, 1, hk, prompt).expand(batch, -1, -1, -1).cuda() for _ in range(2))
    cache = DecodeCache(module, max_tail=tail)
    cache.per, cache.out_dtype = 1, torch.float32
    Prefill(module, bands_fn_of(torch.tensor([[S.INF, S.INF]] * hq, dtype=torch.int32)), cache).store_only(0, k, v, hq)
    e = cache.layers[0]
    assert e["splits"] == splits
    q, kt, vt = (torch.randn(batch, h, n, 128, generator=g).to(torch.bfloat16) for h, n in ((hq, 1), (hk, tail), (hk, tail)))
    token = [x.contiguous().cuda() for x in (q, kt[:, :, -1:], vt[:, :, -1:])]
    e["tail_k"][:, :, :tail - 1], e["tail_v"][:, :, :tail - 1] = kt[:, :, :-1].cuda(), vt[:, :, :-1].cuda()
    cache.step.fill_(tail - 1)
    cache.host_step = tail - 1
    out = cache(0, *token, scale)
    # float64: the partials are relative to the prompt's mean key, as the tail's scores are
    pm, pl, po = (x.double().cpu() for x in e[("partials", hq)])
    pm, pl, po = pm.view(batch, hq, splits), pl.view(batch, hq, splits), po.view(batch, hq, splits, 128)
    mean = e["kstat"][:, :, 0].double().cpu()
    vmean, vscale = e["vstat"][:, :, 0].double().cpu(), e["vstat"][:, :, 1].double().cpu()
    rep = lambda x: x.repeat_interleave(hq // hk, 1)
    s = (rep(kt.double() - mean[:, :, None]) * q.double()).sum(3) * (scale * np.log2(np.e))
    m = torch.maximum(pm.amax(2), s.amax(2))[:, :, None]
    wp, ws = torch.exp2(pm - m), torch.exp2(s - m)
    prompt_o = (wp[..., None] * po).sum(2) * rep(vscale) + (wp * pl).sum(2)[..., None] * rep(vmean)
    want = (prompt_o + (ws[..., None] * rep(vt.double())).sum(2)) / ((wp * pl).sum(2) + ws.sum(2))[..., None]
    err = (out[:, :, 0].cpu().double() - want).abs()
    assert float(err.max()) <= MAX_ABS and float(err.mean()) <= MEAN_ABS, f"max {err.max():.3e} mean {err.mean():.3e}"
    graph = torch.cuda.CUDAGraph()
    cache.begin_capture()
    with torch.cuda.graph(graph):
        again = cache(0, *token, scale)
    cache.end_capture()
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(again, out)
        again.zero_()


@pytest.mark.parametrize("tail, tiles", [(17, 1), (20, 10), (32, 23)])
def test_a_short_tail_merges_alike_on_narrow_and_wide_grids(module, tail, tiles):
    """One sequence alone and among copies of itself that make the grid wide: the same bits (four waves either way, the
    splits summed in one order)."""
    hq, hk, scale, per = 6, 2, 128 ** -0.5, 1
    copies = -(-2 * module.device_cus() // hq)
    print(f"\n[merge] tail {tail}, {tiles} tiles, alone and {copies} times", flush=True)
    g = S.gen(9400 + tail)
    k, v = S.outlier_tensor(g, 1, hk, 64 * tiles).cuda(), S.outlier_tensor(g, 1, hk, 64 * tiles).cuda()
    kt, vt = (torch.randn(1, hk, tail, 128, generator=g).to(torch.bfloat16).cuda() for _ in range(2))
    q = torch.randn(1, hq, 1, 128, generator=g).to(torch.bfloat16).cuda()
    outs = []
    for batch in (1, copies):
        many = lambda x: x.expand(batch, -1, -1, -1).contiguous()
        cache = DecodeCache(module, max_tail=tail)
        cache.per, cache.out_dtype = per, torch.float32
        bands = torch.tensor([[S.INF, S.INF]] * 3 + [[1, S.INF]] * 3, dtype=torch.int32)
        Prefill(module, bands_fn_of(bands), cache).store_only(0, many(k), many(v), hq)
        e = cache.layers[0]
        e["tail_k"][:, :, :tail - 1], e["tail_v"][:, :, :tail - 1] = kt[:, :, :-1], vt[:, :, :-1]
        cache.step.fill_(tail - 1)
        cache.host_step = tail - 1
        outs.append(cache(0, many(q), many(kt[:, :, -1:]), many(vt[:, :, -1:]), scale))
    assert torch.equal(outs[1], outs[0].expand(copies, -1, -1, -1))
