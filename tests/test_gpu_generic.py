"""The generic GEMM variant (any K, any byte alignment of the weights) at the edges of its tiles, against the oracle.

Its sums are fp32 (bf16 matrix instructions on exactly widened codes), so after the bf16 rounding it differs from the
rounded 64-bit result only where that lies within the fp32 error of a rounding boundary: with K <= 2880 terms the error
of a sum is below 2880 * 2^-24 of its absolute terms, well under 2e-4 of the result's scale, against a bf16 step of
2^-8: fewer than 1 in 100 values may differ, each by one step.
"""

import pytest
import torch

from gaudi_kernels import ops
from oracle import block_fp8, synth

pytestmark = pytest.mark.gpu

# the last: 297 workgroups, more than the CUs (four waves each, two partial sums a wave)
SHAPES = [(1, 1, 1), (1, 31, 127), (16, 33, 129), (17, 32, 1000), (33, 65, 1025), (40, 129, 2880), (257, 1030, 1395)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("offset", [0, 1])
def test_generic_edges(m, n, k, half, offset):
    x = synth.activations(m, k, seed=k)
    w, s = synth.weight(n, k, seed=n)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(m))
    ref = block_fp8.reference(x, w, s, native_half=half, bias=bias)
    buf = torch.zeros(n * k + 16, dtype=torch.uint8, device="cuda")
    wd = buf[offset:offset + n * k].view(n, k)
    wd.copy_(w.view(torch.uint8))
    out = torch.full((m + 1, n + 8), -1.0, dtype=torch.bfloat16, device="cuda")
    ops.block_fp8_gemm(x.cuda(), wd, s.cuda(), bias.cuda(), native_half=half, variant="generic", out=out[:m, :n])
    assert bool((out[m] == -1).all()) and bool((out[:, n:] == -1).all())
    y = out[:m, :n].cpu()
    max_rel, mean_rel = block_fp8.parity(y, ref)
    assert max_rel <= block_fp8.MAX_REL_TOL and mean_rel <= block_fp8.MEAN_REL_TOL
    want = ref.to(torch.bfloat16) if ref.dtype != torch.bfloat16 else ref
    assert float((y != want).float().mean()) <= 0.01 or y.numel() < 100


@pytest.mark.parametrize("n,k", [(2880, 2850), (200, 1000)])
@pytest.mark.parametrize("half", [False, True])
def test_generic_rows_do_not_depend_on_the_batch(n, k, half):
    """A token's bits are the same alone, in one block of tokens and at either count of waves a workgroup (N = 2880:
    M = 64 has 180 workgroups, M = 200 has 630)."""
    x = synth.activations(200, k, seed=7).cuda()
    w, s = synth.weight(n, k, seed=8)
    w, s = w.cuda(), s.cuda()
    big = ops.block_fp8_gemm(x, w, s, native_half=half).view(torch.int16)
    for m in (1, 17, 64):
        assert torch.equal(ops.block_fp8_gemm(x[:m], w, s, native_half=half).view(torch.int16), big[:m])


@pytest.mark.parametrize("m", [5, 40])
def test_generic_reads_no_codes_past_k(m):
    """The codes of the last group's columns past K may hold anything, NaN codes included."""
    n, k = 70, 1000
    w, s = synth.weight(n, k, seed=1)
    q, sa = ops.act_quant(synth.activations(m, k, seed=2).cuda())
    y = ops.block_fp8_gemm_q(q, sa, m, w.cuda(), s.cuda())
    q[-1, :, k % 128:] = 0x7F
    assert torch.equal(ops.block_fp8_gemm_q(q, sa, m, w.cuda(), s.cuda()).view(torch.int16), y.view(torch.int16))
