"""Decode batches of 33 .. 48 tokens (three of the layout's four token tiles) equal the first rows of a batch of 64
bit for bit, in every decode shape, weight order and activation layout, and as a K range."""

import pytest
import torch

from gaudi_kernels import ops
from oracle import block_fp8, synth

pytestmark = pytest.mark.gpu


# N per decode shape (16 waves / 8 waves of one and of two weight tiles / 2 waves), with remainders
@pytest.mark.parametrize("n,k", [(500, 2048), (4100, 1152), (6150, 640), (24600, 256)])
@pytest.mark.parametrize("m", [33, 40, 48])
@pytest.mark.parametrize("half", [False, True])
def test_three_token_tiles(m, n, k, half):
    x = synth.activations(64, k, seed=n)
    w, s = synth.weight(n, k, seed=k)
    xd, wd, sd = x.cuda(), w.cuda(), s.cuda()
    pk = ops.pack_weight(wd)
    big = ops.block_fp8_gemm(xd, wd, sd, native_half=half)
    ref = block_fp8.reference(x[m - 1:m], w, s, native_half=half)
    max_rel, mean_rel = block_fp8.parity(big[m - 1:m].cpu(), ref)
    assert max_rel <= block_fp8.MAX_REL_TOL and mean_rel <= block_fp8.MEAN_REL_TOL
    want = big[:m].view(torch.int16)
    for weight in (wd, pk):
        assert torch.equal(ops.block_fp8_gemm(xd[:m], weight, sd, native_half=half).view(torch.int16), want)
        q, sa = ops.act_quant(xd[:m], native_half=half, decode_layout=True)
        y = ops.block_fp8_gemm_q(q, sa, m, weight, sd, native_half=half, decode_layout=True)
        assert torch.equal(y.view(torch.int16), want)
        q, sa = ops.act_quant(xd[:m], native_half=half, m_pad=64)
        assert torch.equal(ops.block_fp8_gemm_q(q, sa, m, weight, sd, native_half=half).view(torch.int16), want)
    part = ops.block_fp8_gemm_kslice(xd[:m], pk, sd, 128, k - 128, native_half=half)
    assert torch.equal(part, ops.block_fp8_gemm_kslice(xd, pk, sd, 128, k - 128, native_half=half)[:m])


# N per decode shape as above; K = 4096 at N = 6150 quantizes inside the kernel up to M = 16
@pytest.mark.parametrize("n,k", [(500, 2048), (4100, 1152), (6150, 4096), (24600, 256)])
@pytest.mark.parametrize("packed", [False, True])
def test_rows_do_not_depend_on_the_batch(n, k, packed):
    x = synth.activations(64, k, seed=n).cuda()
    w, s = synth.weight(n, k, seed=k, device="cuda")
    weight = ops.pack_weight(w) if packed else w
    big = ops.block_fp8_gemm(x, weight, s).view(torch.int16)
    for m in (1, 5, 16, 17, 32, 49):
        assert torch.equal(ops.block_fp8_gemm(x[:m], weight, s).view(torch.int16), big[:m])
