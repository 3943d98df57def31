"""The partial finish's four-column form equals its single-column form and fp32 addition with one bf16 rounding."""

import pytest
import torch

from gaudi_kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,width,pad", [(1, 4, 0), (3, 1028, 0), (70, 260, 4), (2, 1023, 0), (5, 8, 1)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_finish_forms(rows, width, pad, with_bias):
    gen = torch.Generator(device="cuda").manual_seed(rows + width)
    buf = torch.randn(rows, width + pad, device="cuda", generator=gen)
    p = buf[:, :width]
    p[0, 0], p[0, 1], p[0, 2] = float("inf"), float("nan"), -0.0
    b = torch.randn(width + 1, device="cuda", generator=gen)[:width] if with_bias else None
    want = (p if b is None else p + b).bfloat16()
    y = ops.partial_finish(p, b)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    assert torch.equal(torch.nan_to_num(y), torch.nan_to_num(want))
    odd = torch.full((rows, width + 1), 7.0, dtype=torch.bfloat16, device="cuda")  # an odd row stride: single columns
    ops.partial_finish(p, b, out=odd[:, :width])
    assert torch.equal(odd[:, :width].view(torch.int16), y.view(torch.int16)) and bool((odd[:, width] == 7).all())
