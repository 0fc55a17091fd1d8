"""A decode step captured before any eager step of its cache."""
from __future__ import annotations

import pytest
import torch

from helpers import bands_fn_of
from triattention_amd import synthetic as S
from triattention_amd.kernels.decode import DecodeCache
from triattention_amd.kernels.prefill import Prefill

pytestmark = pytest.mark.gpu

SCALE = 128 ** -0.5


def prompt(module, exact, cache=None, seed=9700):
    """A cache holding one 900-token prompt, and its first token."""
    g = S.gen(seed)
    bands = torch.tensor([[S.INF, S.INF]] * 3 + [[1, S.INF]] * 3, dtype=torch.int32)
    k, v = (S.outlier_tensor(g, 1, 2, 900).cuda() for _ in range(2))
    cache = DecodeCache(module, max_tail=8) if cache is None else cache
    Prefill(module, bands_fn_of(bands, exact), cache).store_only(0, k, v, 6)
    return cache, [S.outlier_tensor(g, 1, h, 1).cuda() for h in (6, 2, 2)]


def capture(cache, token, **kw):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, **kw):
        out = cache(0, *token, SCALE)
    return graph, out


@pytest.mark.parametrize("eager_first", [False, True])
def test_a_cache_with_exact_heads_captures_its_first_step(module, eager_first):
    """Captured, it gathers; an eager step, before or after the first replay, runs from its table.  All agree."""
    cache, token = prompt(module, [1])
    want = prompt(module, [1])[0](0, *token, SCALE).clone()
    torch.cuda.synchronize()
    graph, out = capture(cache, token)
    if eager_first:
        assert torch.equal(cache(0, *token, SCALE), want)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        out.zero_()
        assert torch.equal(cache(0, *token, SCALE), want)
    assert "tasks" in cache.layers[0]


@pytest.mark.parametrize("kept", [False, True])
def test_a_quantized_cache_asks_for_an_eager_step_first(module, kept):
    """Also where an earlier prompt of its shape, on the capture's stream, has left the task items (``kept``); the
    eager step that follows finds nothing half built."""
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        cache, token = prompt(module, [], seed=9701)
        if kept:
            cache(0, *token, SCALE)
        cache, token = prompt(module, [], cache)
        fresh, _ = prompt(module, [])
        want = fresh(0, *token, SCALE).clone()
    stream.synchronize()
    with pytest.raises(RuntimeError, match="run one step before capturing"):
        capture(cache, token, stream=stream)
    with torch.cuda.stream(stream):
        assert torch.equal(cache(0, *token, SCALE), want)
        graph, out = capture(cache, token, stream=stream)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
