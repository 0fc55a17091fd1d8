"""GPU parity of the two prepare launches (tri_prepare_qk, tri_pack_v, tri_pack_exact, tri_prepare).

Codes, scales, statistics and records are whole numbers or single correctly rounded operations: every
array is held to the oracle bit for bit, and the one-call form to the three separate calls.  Sizes: one
token, either side of a tile, prompts whose record workgroups take one tile each and several (a head's
last workgroup then takes fewer), statistics chains of one load batch, two and a remainder; inputs
token-major (as HF projections give them), head-major, and a padded row stride.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from helpers import compare_codes
from triattention_amd import synthetic as S
from triattention_amd.kernels.prefill import F16, I4, I8, Layout, Prefill, Q4
from triattention_amd.maps import uniform
from triattention_amd.synthetic import bits

pytestmark = pytest.mark.gpu


def on_device(x, layout):
    """x [B, H, T, 128] on the GPU in the named memory layout."""
    b, h, t, d = x.shape
    if layout == "head":
        return x.cuda()
    pad = 4 if layout == "padded" else 0  # rows 8-byte aligned only
    y = torch.full((b, t, h, d + pad), float("nan"), dtype=x.dtype, device="cuda")
    y[..., :d] = x.transpose(1, 2).cuda()
    return y[..., :d].transpose(1, 2)


@pytest.mark.parametrize("batch, hq, hk, t, layout", [
    (1, 6, 2, 1, "head"), (2, 3, 3, 64, "token"), (1, 4, 2, 65, "padded"), (1, 2, 1, 1025, "token"),
    (2, 4, 4, 8193, "head"), (3, 8, 8, 3001, "padded")])
def test_prepare_matches_the_oracle_and_the_separate_calls(module, batch, hq, hk, t, layout):
    print(f"\n[prepare] batch={batch} hq={hq} hk={hk} t={t} {layout}", flush=True)
    g = S.gen(7000 + t)
    host = [S.outlier_tensor(g, batch, h, t) for h in (hq, hk, hk)]
    q, k, v = (on_device(x, layout) for x in host)
    lay = Layout(batch, hq, hk, t, True, frozenset((F16, I8, I4, Q4)))
    pres = [Prefill(module, uniform(1, 2)) for _ in range(2)]
    ops, sep = (p.operands(lay, q.device) for p in pres)
    for x in list(ops.values()) + list(ops["packed"].values()) + list(sep.values()) + list(sep["packed"].values()):
        if isinstance(x, torch.Tensor):
            x.view(torch.uint8).fill_(0xA5)
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
    bands = np.array([[1, 1 << 20]] * hq)
    for b in range(batch):
        codes = O.prefill_codes(*(bits(x[b]) for x in host), bands, decode_cache=t > 1088)
        if codes["v4"] is None:  # (short prompts keep no INT4 V: pack it from the same statistics)
            codes["v4"] = O.pack_v(bits(host[2][b]), codes["vstat"], True, True, True)[2]
        if not codes["identity"]:
            compare_codes(ops, codes, b, batch, hq, hk, t)


@pytest.mark.parametrize("t, flags", [(1, [1, 0]), (130, [0, 1]), (130, [2, 1])])
def test_prepare_writes_the_exact_records(module, t, flags):
    """The exact heads' KX / VX records of the one-call form equal pack_exact's; a quantized head's are
    left alone."""
    g = S.gen(7100 + t)
    q, k, v = (S.outlier_tensor(g, 2, h, t).cuda() for h in (4, 2, 2))
    tiles, nx = (t + 63) // 64, max(flags)
    exact = torch.tensor([f for f in flags for _ in range(2)], dtype=torch.int32, device="cuda")
    pre = Prefill(module, uniform(1, 2))
    ops = pre.operands(Layout(2, 4, 2, t, False, frozenset((F16,))), q.device)
    out = [torch.full((2 * nx * tiles * 16384,), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(4)]
    module.prepare(q, k, v, ops["q8"], ops["qa"], ops["kp"], ops["ka"], ops["partial"], ops["kstat"], None, None, None,
                   None, None, ops["vpartial"], ops["vstat"], ops["packed"][F16], None, None, None, exact, nx, *out[:2])
    module.pack_exact(k, v, exact, nx, *out[2:])
    assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[3])
    assert bool((ops["vstat"][:, :, 0] == 0).all()) and bool((ops["vstat"][:, :, 1:] == 1).all())  # identity V
