"""GPU parity of the prepare launches (tri_prepare_qk, tri_pack_v, tri_pack_exact, tri_prepare).

Codes, scales, statistics and records are whole numbers or single correctly rounded operations: every
array is held to the oracle bit for bit at every size, the expanded INT4 keys and the V8 sums to the records
they come from, the exact heads' records to a host packing of the documented layout, and the one-call form to
the three separate calls.  The bytes past each buffer stay as they were.  Sizes: one
token, either side of a tile, prompts whose record workgroups take one tile each and several (a head's
last workgroup then takes fewer), statistics chains of one load batch, two and a remainder; inputs
token-major (as HF projections give them), head-major, and a padded row stride.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from cache_host import pack_kx
from helpers import compare_codes
from triattention_amd import synthetic as S
from triattention_amd.kernels import records as R
from triattention_amd.kernels.prefill import F16, I4, I8, Layout, Prefill, Q4
from triattention_amd.maps import uniform
from triattention_amd.synthetic import bits

pytestmark = pytest.mark.gpu

GUARD, FILL = 4096, 0xA5  # bytes past each buffer, and what every byte holds before the calls


def on_device(x, layout):
    """x [B, H, T, 128] on the GPU in the named memory layout."""
    b, h, t, d = x.shape
    if layout == "head":
        return x.cuda()
    pad = 4 if layout == "padded" else 0  # rows 8-byte aligned only
    y = torch.full((b, t, h, d + pad), float("nan"), dtype=x.dtype, device="cuda")
    y[..., :d] = x.transpose(1, 2).cuda()
    return y[..., :d].transpose(1, 2)


def guarded(module, lay, device):
    """A prompt's operands in a scratch of their sizes plus GUARD bytes, every byte FILL; and a check that
    those bytes still are."""
    sizes, pre = Prefill(module, uniform(1, 2)), Prefill(module, uniform(1, 2))
    sizes.operands(lay, device)
    for name, x in sizes.buffers.items():
        pool = torch.full((x.numel() * x.element_size() + GUARD,), FILL, dtype=torch.uint8, device=device)
        pre.buffers[name] = pool.view(x.dtype)

    def check():
        for name, x in pre.buffers.items():
            n = sizes.buffers[name].numel() * x.element_size()
            assert bool((x.view(torch.uint8)[n:] == FILL).all()), f"written past {name}"
    return pre.operands(lay, device), check


def all_codes(q, k, v):
    """The oracle's operands of one sequence with every format, whatever a map of this length would keep."""
    _, kstat = O.stats(k)
    _, vstat = O.stats(v)
    names = ("q8", "qa", "q4", "qa4", "k8", "ka", "k4", "ka4", "v16", "v8", "v4")
    codes = dict(zip(names, O.quantize_q(q, True) + O.quantize_k(k, kstat, True) + O.pack_v(v, vstat)))
    return dict(codes, kstat=kstat, vstat=vstat)


@pytest.mark.parametrize("batch, hq, hk, t, layout", [
    (1, 6, 2, 1, "head"), (2, 3, 3, 64, "token"), (1, 4, 2, 65, "padded"), (1, 2, 1, 1025, "token"),
    (2, 4, 4, 8193, "head"), (3, 8, 8, 3001, "padded"),
    # either side of the sizes whose statistics a launch of their own completes: no call, the one call, the one call
    # and pack_v, all three
    (10, 2, 2, 380, "padded"), (10, 2, 2, 450, "token"), (14, 2, 2, 300, "head"), (40, 2, 2, 450, "token")])
def test_prepare_matches_the_oracle_and_the_separate_calls(module, batch, hq, hk, t, layout):
    print(f"\n[prepare] batch={batch} hq={hq} hk={hk} t={t} {layout}", flush=True)
    g = S.gen(7000 + t)
    host = [S.outlier_tensor(g, batch, h, t) for h in (hq, hk, hk)]
    q, k, v = (on_device(x, layout) for x in host)
    lay = Layout(batch, hq, hk, t, True, frozenset((F16, I8, I4, Q4)))
    (ops, past), (sep, past_sep) = (guarded(module, lay, q.device) for _ in range(2))
    p, s = ops["packed"], sep["packed"]
    module.prepare(q, k, v, ops["q8"], ops["qa"], ops["kp"], ops["ka"], ops["partial"], ops["kstat"], ops["q4"],
                   ops["qa4"], ops["k4"], ops["ka4"], ops["k4x"], ops["vpartial"], ops["vstat"], p[F16], p[I8], p[I4],
                   ops["v8sum"])
    module.prepare_qk(q, k, sep["q8"], sep["qa"], sep["kp"], sep["ka"], sep["partial"], sep["kstat"], sep["q4"],
                      sep["qa4"], sep["k4"], sep["ka4"], k4x=sep["k4x"])
    module.pack_v(v, sep["partial"], sep["vstat"], s[F16], s[I8], s[I4], v8sum=sep["v8sum"])
    torch.cuda.synchronize()
    for name in ("q8", "qa", "kp", "ka", "kstat", "q4", "qa4", "k4", "ka4", "k4x", "vstat", "v8sum"):
        assert torch.equal(ops[name].view(torch.uint8), sep[name].view(torch.uint8)), name
    for code in (F16, I8, I4):
        assert torch.equal(p[code].view(torch.uint8), s[code].view(torch.uint8)), code
    past()
    past_sep()
    tiles = (t + 63) // 64
    k4x = R.unpack_k8(ops["k4x"].cpu().numpy()).reshape(batch, hk, tiles * 64, 128)
    sums = ops["v8sum"].cpu().numpy().reshape(batch, hk, tiles, 128)
    for b in range(batch):
        codes = all_codes(*(bits(x[b]) for x in host))
        compare_codes(ops, codes, b, batch, hq, hk, t)
        np.testing.assert_array_equal(k4x[b].astype(np.int32), 16 * codes["k4"].astype(np.int32))
        np.testing.assert_array_equal(sums[b], -127 * codes["v8"].reshape(hk, tiles, 64, 128).sum(2, dtype=np.int32))


@pytest.mark.parametrize("t", [1, 64, 65])
def test_prepare_without_quantized_v_keeps_it(module, t):
    """With V16 records alone V' is V itself: the statistics are (0, 1, 1), the records V's fp16 values."""
    g = S.gen(7050 + t)
    host = [S.outlier_tensor(g, 2, h, t) for h in (4, 2, 2)]
    q, k, v = (x.cuda() for x in host)
    ops, past = guarded(module, Layout(2, 4, 2, t, False, frozenset((F16,))), q.device)
    module.prepare(q, k, v, ops["q8"], ops["qa"], ops["kp"], ops["ka"], ops["partial"], ops["kstat"], None, None, None,
                   None, None, ops["vpartial"], ops["vstat"], ops["packed"][F16], None, None, None)
    past()
    for b in range(2):
        codes = O.prefill_codes(*(bits(x[b]) for x in host), np.array([[9, 9]] * 4))
        assert codes["identity"] and codes["k4"] is None and codes["v8"] is None
        compare_codes(ops, codes, b, 2, 4, 2, t)


@pytest.mark.parametrize("t, flags", [(1, [1, 0]), (64, [0, 1]), (65, [0, 1, 2]), (130, [0, 1]), (130, [2, 1])])
def test_prepare_writes_the_exact_records(module, t, flags):
    """The exact heads' KX / VX records of the one-call form and of pack_exact are the documented layout's,
    zeros past the prompt; nothing is written for a quantized head, nor outside the records."""
    g = S.gen(7100 + t)
    batch, hk, hq = 2, len(flags), 2 * len(flags)
    host = [S.outlier_tensor(g, batch, h, t) for h in (hq, hk, hk)]
    q, k, v = (x.cuda() for x in host)
    tiles, nx = (t + 63) // 64, max(flags)
    exact = torch.tensor([f for f in flags for _ in range(2)], dtype=torch.int32, device="cuda")
    ops, past = guarded(module, Layout(batch, hq, hk, t, False, frozenset((F16,))), q.device)
    # (a head's records of guard on either side: a quantized head has slot -1)
    n, guard = batch * nx * tiles * 16384, tiles * 16384
    out = [torch.full((n + 2 * guard,), FILL, dtype=torch.uint8, device="cuda") for _ in range(4)]
    kx, vx, kx2, vx2 = (x[guard:guard + n] for x in out)
    module.prepare(q, k, v, ops["q8"], ops["qa"], ops["kp"], ops["ka"], ops["partial"], ops["kstat"], None, None, None,
                   None, None, ops["vpartial"], ops["vstat"], ops["packed"][F16], None, None, None, exact, nx, kx, vx)
    module.pack_exact(k, v, exact, nx, kx2, vx2)
    past()
    want = np.zeros((2, batch, nx, tiles, 16384), np.uint8)
    rows = np.zeros((2, batch, hk, tiles * 64, 128), np.uint16)
    for i, x in enumerate(host[1:]):
        rows[i, :, :, :t] = bits(x)
    for h, f in enumerate(flags):
        for b in range(batch if f else 0):
            for j in range(tiles):
                want[:, b, f - 1, j] = pack_kx(*rows[:, b, h, 64 * j:64 * j + 64])
    for i, x in enumerate(out):
        got = x.cpu().numpy()
        np.testing.assert_array_equal(got[guard:guard + n], want[i % 2].reshape(-1))
        assert (got[:guard] == FILL).all() and (got[guard + n:] == FILL).all()
    assert bool((ops["vstat"][:, :, 0] == 0).all()) and bool((ops["vstat"][:, :, 1:] == 1).all())  # identity V


def test_prepare_qk_past_one_grid(module):
    """65,535 one-token sequences of 257 q-heads: 17.9 million workgroups, more than one grid holds.  Every row
    holds its sequence's codes, as the same sequences with one q-head in one grid give them."""
    batch, heads = 65535, 257
    g = torch.Generator(device="cuda").manual_seed(7200)
    q, k = (torch.randn(batch, 1, 1, 128, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    new = lambda *shape, dtype=torch.float32: torch.full(shape, 7, dtype=dtype, device="cuda")
    kp, partial, outs = new(batch * 2048, dtype=torch.int32), new(batch * 64 * 3 * 128), []
    for h in (1, heads):
        q8, qa, ka, kstat = new(batch, h, 1, 128, dtype=torch.int8), new(batch * h), new(batch * 4), new(batch * 3 * 128)
        print(f"\n[prepare] {batch} sequences of one token, {h} q-heads", flush=True)
        module.prepare_qk(q.expand(-1, h, -1, -1), k, q8, qa, kp.view(torch.uint32), ka, partial, kstat)
        outs.append((q8.view(batch, h, 128), qa.view(batch, h), ka, kstat, kp.clone()))
    one, many = outs
    for b in range(0, batch, 4096):  # (a slice at a time: the comparison's temporaries stay small)
        assert bool((many[0][b:b + 4096] == one[0][b:b + 4096]).all())
    assert bool((many[1] == one[1]).all())
    assert all(torch.equal(x, y) for x, y in zip(one[2:], many[2:]))
    codes = O.quantize_q(bits(q[:64, 0].cpu()), False)  # [64 rows as heads, one token]
    np.testing.assert_array_equal(one[0][:64, 0].cpu().numpy(), codes[0][:, 0])
