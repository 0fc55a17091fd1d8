"""Which launch form the size-based choice of ``tri_attention`` takes on both sides of its lines.

Its output equals the expected form's bit for bit (the forms differ in summation order, so the other
form's differs).  Both are convex combinations of V's rows from the same probabilities, summed in fp32 a
tile at a time: each tile's add and rescale rounds twice, at most 2**-24 of max|V| each time, per form."""
from __future__ import annotations

import pytest
import torch

from helpers import bands_fn_of
from triattention_amd import synthetic as S
from triattention_amd.kernels.prefill import Prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch, hq, hk, t, exact, form", [
    (1, 24, 8, 1344, [], 2),      # 504 workgroups: two per CU or fewer
    (1, 24, 8, 1400, [], 2),      # 528: few rows
    (1, 24, 8, 1400, [1], 1),     # exact heads beyond two per CU
    (1, 32, 8, 2047, [], 2),      # 1,024, batch * hq = CUs / 8
    (1, 32, 8, 2049, [], 1),      # 1,056
    (2, 14, 2, 1100, [], 2),      # 504 in two sequences
    (2, 14, 2, 1300, [], 2),      # 588 in two sequences
    (1, 36, 4, 1300, [], 1),      # 756 in more rows than CUs / 8
    (4, 24, 8, 512, [], 1)])      # 768 in 96 rows
def test_the_choice_by_size(module, batch, hq, hk, t, exact, form):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are those of 256 CUs")
    g = S.gen(9600 + t + hq)
    q, k, v = (S.outlier_tensor(g, batch, h, t).cuda() for h in (hq, hk, hk))
    bands = torch.tensor([[1, S.INF] if (r * hk // hq) % 2 else [S.INF, S.INF] for r in range(hq)], dtype=torch.int32)
    outs = {}
    try:
        for mode in (1, 2, 0):
            module.prefill_pairs(mode)
            pre = Prefill(module, bands_fn_of(bands, exact), out_dtype=torch.float32)
            outs[mode] = pre(0, q, k, v, 128 ** -0.5).clone()
    finally:
        module.prefill_pairs(0)
    assert torch.equal(outs[0], outs[form])
    assert not torch.equal(outs[1], outs[2])
    assert (outs[1] - outs[2]).abs().max() <= 4 * ((t + 63) // 64) * 2 ** -24 * v.float().abs().max()
