"""Every bf16 gate through SiLU-and-mul (up = 1) against the 64-bit value, and the same bits whichever of the kernel's
two forms a gate's neighbours select."""

import pytest
import torch

from gaudi_kernels import ops

pytestmark = pytest.mark.gpu


def _all_gates():
    g = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    return g[torch.isfinite(g.float())]


def test_every_gate_against_64_bits():
    """silu is a few fp32 roundings (2 ulps, 2^-22) and one bf16 rounding: at most one bf16 step from the rounded
    64-bit value, and only where that lies within 2^-22 of a rounding boundary (about 2^-13 of the values)."""
    g = _all_gates()
    x = torch.cat([g, torch.ones_like(g)]).view(1, -1).cuda()
    y = ops.silu_and_mul(x)[0].cpu()
    v = g.double()
    want = torch.where(v <= -88, torch.zeros_like(v), v / (1 + torch.exp(-v))).float().bfloat16()
    step = (y.view(torch.int16).int() - want.view(torch.int16).int()).abs()
    assert int(step.max()) <= 1
    assert float((step != 0).float().mean()) <= 2.0 ** -12


@pytest.mark.parametrize("quant", [False, True])
def test_neighbours_do_not_matter(quant):
    g = _all_gates()
    g = g[g.float().abs() <= 80][: 65536 // 128 * 64]
    g = g[: g.numel() // 128 * 128]
    u = torch.linspace(-2, 2, g.numel()).bfloat16()
    rows = g.numel() // 128
    gate, up = g.view(rows, 128).clone(), u.view(rows, 128).clone()
    y = ops.silu_and_mul(torch.cat([gate, up], 1).cuda())
    gate[:, ::8], up[:, 1::8] = 100.0, float("inf")  # one gate out of range, one infinite up value in every eight
    z = ops.silu_and_mul(torch.cat([gate, up], 1).cuda())
    keep = torch.ones(128, dtype=torch.bool)
    keep[::8] = keep[1::8] = False
    assert torch.equal(y[:, keep].view(torch.int16), z[:, keep].view(torch.int16))
    if quant:
        gate[:, ::8], up[:, 1::8] = 100.0, 3.0
        x = torch.cat([gate, up], 1).cuda()
        q, s = ops.silu_mul_quant(x)
        q2, s2 = ops.act_quant(ops.silu_and_mul(x))
        assert torch.equal(q, q2) and torch.equal(s, s2)
