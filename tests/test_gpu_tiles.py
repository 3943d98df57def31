"""The mid-sized tiles of the LDS-tiled GEMM (csrc/gk_fp8_tiles.hip) against the oracle and against the 256 x 256 kernel.

A token's output does not depend on the other tokens, and every tile adds the groups in the same order, so the first
rows of a product that the 256 x 256 kernel computes (M = 4096) equal the small product bit for bit.  The shapes reach
every tile of plan_tile (test_tiles_host.py checks that), each with a remainder of its rows, columns or groups.
"""

import pytest
import torch

from gaudi_kernels import ops
from oracle import block_fp8, synth

pytestmark = pytest.mark.gpu

# (m, n, k): 64x32, 64x64, 128x64, 128x64 twice a CU, 128x128
SHAPES = [(65, 500, 384), (128, 6140, 640), (300, 6144, 640), (777, 5003, 384), (1000, 4090, 896)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("half", [False, True])
def test_tiles_against_oracle(m, n, k, half):
    x = synth.activations(m, k, seed=m)
    w, s = synth.weight(n, k, seed=n)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(k))
    rows = sorted({0, 1, m // 2, m - 2, m - 1})
    ref = block_fp8.reference(x[rows], w, s, native_half=half, bias=bias)
    wd, sd, bd = w.cuda(), s.cuda(), bias.cuda()
    outs = []
    for weight in (wd, ops.pack_weight(wd)):
        out = torch.full((m + 1, n + 8), -1.0, dtype=torch.bfloat16, device="cuda")
        ops.block_fp8_gemm(x.cuda(), weight, sd, bd, native_half=half, out=out[:m, :n])
        assert bool((out[m] == -1).all()) and bool((out[:, n:] == -1).all())  # only inside [M, N]
        outs.append(out[:m, :n].clone())
    max_rel, mean_rel = block_fp8.parity(outs[0][rows].cpu(), ref)
    assert max_rel <= block_fp8.MAX_REL_TOL and mean_rel <= block_fp8.MEAN_REL_TOL
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("m,n,k", [(65, 6144, 256), (300, 6144, 8320), (128, 6144, 384), (1024, 6144, 128)])
def test_tiles_equal_256_rows(m, n, k):
    """k = 8320: 65 groups, past one register of weight scales."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    x = torch.randn(4096, k, generator=gen, device="cuda").bfloat16()
    w, s = synth.weight(n, k, seed=3, device="cuda")
    big = ops.block_fp8_gemm(x, w, s)
    assert torch.equal(ops.block_fp8_gemm(x[:m], w, s).view(torch.int16), big[:m].view(torch.int16))


# 64x32, 64x64, 128x64, 128x64 twice a CU (two), 128x128, 256x256 in one range and (last) in two of 256 and 192 columns
@pytest.mark.parametrize("m,n,k", [(17, 500, 384), (128, 6140, 640), (300, 6144, 256), (777, 5003, 384),
                                   (1000, 4090, 128), (640, 4090, 2048), (2047, 7168, 256), (4095, 7160, 256)])
def test_channel_tiles(m, n, k):
    """Every tile of the per-channel GEMM against 64-bit products: P is a sum of at most 2048 exact products whose
    fp8 matrix instruction sums to within 1e-4 of its scale; the rest is three fp32 roundings and the bf16 one."""
    gen = torch.Generator(device="cuda").manual_seed(m)
    q, sa = ops.token_quant(torch.randn(m, k, generator=gen, device="cuda").bfloat16())
    w = torch.randint(0, 127, (n, k), dtype=torch.uint8, device="cuda", generator=gen)
    w |= torch.randint(0, 2, (n, k), dtype=torch.uint8, device="cuda", generator=gen) << 7
    sw, bias = torch.rand(n, device="cuda", generator=gen), torch.randn(n, device="cuda", generator=gen)
    out = torch.full((m + 1, n + 8), -1.0, dtype=torch.bfloat16, device="cuda")
    ops.channel_gemm(q, sa, w, sw, bias, out=out[:m, :n])
    assert bool((out[m] == -1).all()) and bool((out[:, n:] == -1).all())
    a = q.view(torch.float8_e4m3fn).double()
    p = (a @ w.view(torch.float8_e4m3fn).double().t()) * sa.double()[:, None] * sw.double()
    scale = (a.abs() @ w.view(torch.float8_e4m3fn).double().abs().t()) * sa.double()[:, None] * sw.double()
    err = (out[:m, :n].double() - (p + bias.double())).abs()
    assert bool((err <= 2.0 ** -8 * (p + bias.double()).abs() + 1e-4 * scale + 1e-6).all())
    odd = torch.empty(m, n + 1, dtype=torch.bfloat16, device="cuda")[:, :n]  # rows that take no wide stores
    ops.channel_gemm(q, sa, w, sw, bias, out=odd)
    assert torch.equal(odd.view(torch.int16), out[:m, :n].view(torch.int16))


@pytest.mark.parametrize("m,n,k", [(65, 500, 384), (300, 6144, 256), (1000, 4090, 128)])
def test_token_scales_aligned_to_four_bytes(m, n, k):
    """Quantized activations whose scales start one float into a buffer: the same bits as aligned ones."""
    w, s = synth.weight(n, k, seed=3, device="cuda")
    q, sa = ops.act_quant(synth.activations(m, k, seed=4).cuda(), m_pad=ops.plan(m, n, k)[1])
    odd = torch.empty(sa.numel() + 1, device="cuda")[1:].view_as(sa).copy_(sa)
    assert odd.data_ptr() % 16 == 4 and odd.is_contiguous()
    want = ops.block_fp8_gemm_q(q, sa, m, w, s).view(torch.int16)
    assert torch.equal(ops.block_fp8_gemm_q(q, odd, m, w, s).view(torch.int16), want)
