"""A prompt whose KV heads are all exact refuses what the quantized path's preparation refuses."""
from __future__ import annotations

import pytest
import torch

from helpers import bands_fn_of
from triattention_amd import synthetic as S
from triattention_amd.kernels.extension import Module, load_library
from triattention_amd.kernels.prefill import Prefill

EXACT = bands_fn_of(torch.tensor([[S.INF, S.INF]] * 4, dtype=torch.int32), [0, 1])


def zeros(*shape, device, dtype=torch.bfloat16):
    return torch.zeros(shape, device=device, dtype=dtype)


def test_operands_off_the_gpu_are_refused():
    kv = zeros(1, 2, 70, 128, device="cpu")
    with pytest.raises(RuntimeError, match="BF16 Q/K"):
        Prefill(Module(load_library()), EXACT)(0, zeros(1, 4, 70, 128, device="cpu"), kv, kv, 1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("q, k", [((1, 4, 70, 128), (1, 2, 69, 128)), ((1, 4, 70, 128), (1, 2, 130, 128)),
                                  ((2, 4, 70, 128), (1, 2, 70, 128)), ((1, 4, 70, 64), (1, 2, 70, 128))])
def test_queries_and_keys_of_other_shapes_are_refused(module, q, k):
    kv = zeros(*k, device="cuda")
    with pytest.raises(RuntimeError, match="BF16 Q/K"):
        Prefill(module, EXACT)(0, zeros(*q, device="cuda"), kv, kv, 1.0)


@pytest.mark.gpu
def test_tensors_on_the_host_are_refused(module):
    q, kv = zeros(1, 4, 70, 128, device="cuda"), zeros(1, 2, 70, 128, device="cuda")
    with pytest.raises(RuntimeError):
        Prefill(module, EXACT)(0, q, kv.cpu(), kv.cpu(), 1.0)
