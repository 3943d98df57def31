"""RMSNorm of few rows (512 or 1024 threads a row beyond 2048 columns) equals the first rows of a large batch (256
threads a row) bit for bit, at the edges of the widths where the thread count changes."""

import pytest
import torch

from gaudi_kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [2048, 2049, 4096, 4104, 8191, 8192])
def test_few_rows_equal_many(width):
    gen = torch.Generator(device="cuda").manual_seed(width)
    x = torch.randn(300, width, device="cuda", generator=gen).bfloat16()
    r = torch.randn(300, width, device="cuda", generator=gen).bfloat16()
    g = torch.randn(width, device="cuda", generator=gen).bfloat16()
    assert torch.equal(ops.rms_norm(x[:5], g).view(torch.int16), ops.rms_norm(x, g)[:5].view(torch.int16))
    few, many = ops.fused_add_rms_norm(x[:5], r[:5], g), ops.fused_add_rms_norm(x, r, g)
    for a, b in zip(few, many):
        assert torch.equal(a.view(torch.int16), b[:5].view(torch.int16))
    q, sa, res = ops.rms_norm_quant(x[:5], g, residual=r[:5])
    q2, sa2, res2 = ops.rms_norm_quant(x, g, residual=r)
    assert torch.equal(q, q2[:, :5]) and torch.equal(sa, sa2[:, :5])
    assert torch.equal(res.view(torch.int16), res2[:5].view(torch.int16))
