"""RMSNorm of few rows (512 or 1024 threads a row beyond 2048 columns) equals the first rows of a large batch (256
threads a row) bit for bit, at the edges of the widths where the thread count changes."""

import math

import pytest
import torch

from gaudi_kernels import ops
from oracle import norm

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


@pytest.mark.parametrize("width", [2064, 4096, 8192])
def test_sums_that_depend_on_the_order(width):
    """Rows whose fp64 sum of squares ends beside the middle of two fp32 values, on the side that the order of 256
    threads gives: 1 + 2^-24 absorbs eight squares of 2^-54 one by one, their own sum of 2^-51 it does not."""
    gen = torch.Generator().manual_seed(0)
    x = torch.randint(-32, 33, (200, width), generator=gen).float() * 2.0 ** -11
    x[:, 0], x[:, 1], x[:, 2048:2056] = 1.0, 2.0 ** -12, 2.0 ** -27
    x, g = x.bfloat16(), torch.randn(width, generator=gen).bfloat16()
    exact = torch.tensor([math.fsum((r.double() ** 2).tolist()) for r in x]).float()
    assert not bool((exact == torch.from_numpy(norm.sum_squares(x))).any())
    want = norm.rms_norm(x, g, 1e-30)
    xd, gd, zero = x.cuda(), g.cuda(), torch.zeros_like(x).cuda()
    y = ops.rms_norm(xd, gd, 1e-30)
    assert torch.equal(y.cpu().view(torch.int16), want.view(torch.int16))
    res, y = ops.fused_add_rms_norm(zero, xd, gd, 1e-30)
    assert torch.equal(y.cpu().view(torch.int16), want.view(torch.int16)) and torch.equal(res, xd)
    q, sa = ops.act_quant(want.cuda())
    q2, sa2, _ = ops.rms_norm_quant(zero, gd, 1e-30, residual=xd)
    assert torch.equal(q2, q) and torch.equal(sa2, sa)
