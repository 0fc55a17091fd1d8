"""Host tensors never reach a kernel: every entry point refuses them before it calls the library.

The library is replaced by one that only records calls, and tensors said to be on the GPU are host tensors
that claim its device, so the checks run where there is no GPU."""
from __future__ import annotations

import types

import pytest
import torch

from helpers import bands_fn_of
from triattention_amd import synthetic as S
from triattention_amd.kernels.extension import KX_BYTES, Module
from triattention_amd.kernels.prefill import Prefill

GPU, OTHER = torch.device("cuda", 0), torch.device("cuda", 1)


class OnGpu(torch.Tensor):
    """A host tensor that claims to be on the GPU."""
    __torch_function__ = torch._C._disabled_torch_function_impl
    is_cuda = property(lambda self: True)
    device = property(lambda self: GPU)

    def get_device(self):
        return self.device.index


class OnOther(OnGpu):
    """The same on another GPU."""
    device = property(lambda self: OTHER)


class Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *args: self.calls.append(name) or 0


@pytest.fixture
def module(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: types.SimpleNamespace(cuda_stream=0))
    return Module(Recorder())


def gpu(t):
    return t.as_subclass(OnGpu)


def i32(*s):
    return torch.zeros(*s, dtype=torch.int32)


def u32(n):
    return i32(n).view(torch.uint32)


def attention(module, wrap):
    return module.attention(wrap(i32(4)), wrap(torch.tensor([[9, 9]] * 4, dtype=torch.int32)), None, None,
                            wrap(u32(2 * 4096)), wrap(u32(2 * 2048)), None, wrap(torch.zeros(1, 2, 3, 128)),
                            wrap(torch.zeros(1, 4, 64, 128, dtype=torch.int8)), wrap(u32(2 * 2048)),
                            wrap(torch.zeros(4 * 64)), wrap(torch.zeros(8)), None, None, None, None,
                            wrap(torch.zeros(1, 4, 64, 128)), 0.1)


def pack_exact(module, wrap):
    kv = wrap(torch.zeros(1, 2, 64, 128, dtype=torch.bfloat16))
    rec = wrap(torch.zeros(KX_BYTES, dtype=torch.uint8))
    module.pack_exact(kv, kv, gpu(torch.tensor([1, 1, 0, 0], dtype=torch.int32)), 1, rec, rec)


def decode_tasks(module, wrap):
    meta = [wrap(i32(1, 2, 3)) for _ in range(3)]
    module.decode_tasks(wrap(torch.zeros(2 * 3 * 4)), None, meta[0], meta[1], wrap(i32(1, 2)), wrap(i32(1, 3)),
                        meta[2], 2)


def cache_store(module, wrap):
    rec = lambda words: wrap(u32(2 * words).view(2, words))
    row = lambda *s, dtype=torch.int32: wrap(torch.zeros(1, 2, *s, dtype=dtype))
    stat = lambda: row(3, 128, dtype=torch.float32)
    dst = dict(entry=row(1), kinfo=row(1), slot=row(1), count=row(), fmt=wrap(i32(1, 1)), prompt=wrap(i32(1)),
               xslot=None, ka=row(1, 4, dtype=torch.float32), ka4=None, kstat=stat(), vstat=stat(), k8=rec(2048),
               k4=None, v8=rec(2048), v4=None, kx=None, vx=None)
    zero = dict(k8=0, k4=0, v8=0, v4=0, x=0)
    module.cache_store(gpu(i32(4, 2)), None, 64, rec(2048), None, row(1, 4, dtype=torch.float32), None, stat(), stat(),
                       rec(2048), None, None, None, 0, 0, dst, zero, dict(zero, k8=2, v8=2))


@pytest.mark.parametrize("entry", [attention, pack_exact, decode_tasks, cache_store])
def test_host_tensors_are_refused(module, monkeypatch, entry):
    empty = torch.empty
    with pytest.raises(ValueError, match="Expected a cuda device"):
        entry(module, lambda t: t)
    assert module.lib.calls == []
    # the same call with device tensors launches once
    monkeypatch.setattr(torch, "empty", lambda *a, device=None, **kw: empty(*a, **kw))
    entry(module, gpu)
    assert len(module.lib.calls) == 1


@pytest.mark.parametrize("exact", [[], [1], [0, 1]])
@pytest.mark.parametrize("place", [lambda t: t, lambda t: t.as_subclass(OnOther)])
@pytest.mark.parametrize("which", ["k", "v"])
def test_a_prompt_on_two_devices_is_refused(module, monkeypatch, exact, place, which):
    """Q, K and V go to one launch as raw addresses, whatever the map keeps quantized or exact."""
    empty, to = torch.empty, torch.Tensor.to
    monkeypatch.setattr(torch, "empty", lambda *a, device=None, **kw: empty(*a, **kw))
    monkeypatch.setattr(torch.Tensor, "to", lambda t, d, *a: gpu(t) if d == GPU else to(t, d, *a))
    x = lambda h: torch.zeros(1, h, 70, 128, dtype=torch.bfloat16)
    qkv = dict(q=gpu(x(4)), k=gpu(x(2)), v=gpu(x(2)))
    bands = torch.tensor([[S.INF, S.INF], [1, S.INF], [S.INF, S.INF], [1, S.INF]], dtype=torch.int32)
    prefill = Prefill(module, bands_fn_of(bands, exact))
    with pytest.raises(RuntimeError, match="on one device|BF16 V"):
        prefill(0, **dict(qkv, **{which: place(x(2))}), scale=0.1)
    assert module.lib.calls == []
    with pytest.raises(RuntimeError, match="on one device"):
        rec = gpu(torch.zeros(4 * KX_BYTES, dtype=torch.uint8))
        kv = {n: qkv[n] for n in "kv"}
        module.pack_exact(**dict(kv, **{which: place(x(2))}), exact=gpu(i32(4)), nx=1, kx=rec, vx=rec)
    assert module.lib.calls == []
    # on one device the prompt is prepared (its attention then finds the stand-in scratch on the host)
    with pytest.raises(ValueError, match="Expected a cuda device"):
        prefill(0, **qkv, scale=0.1)
    assert module.lib.calls == ["tri_pack_exact" if len(exact) == 2 else "tri_prepare"]
