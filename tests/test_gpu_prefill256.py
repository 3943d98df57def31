"""The 256 x 256 kernel (csrc/gk_fp8_prefill.hip) at shapes that it serves itself, in one column range and in two:
its three output forms, and fp32 partials of K ranges summed in place.  test_tiles_host.py checks that these shapes
stay with it for aligned and unaligned rows and for every K range."""

import pytest
import torch

from gaudi_kernels import ops
from oracle import block_fp8, synth

pytestmark = pytest.mark.gpu

SHAPES = [(2040, 7163), (3000, 6001)]  # 224 tiles in one range; 288, so 2048 columns in 256-wide tiles, the rest in 192-wide
K = 1152
RANGES = ((0, 256), (256, 384), (640, 512))
SENTINEL = 0x7E7E  # bf16 bit pattern never produced by these inputs


def _operands(m, n):
    w, s = synth.weight(n, K, seed=n)
    x = synth.activations(m, K, seed=m)
    return x, w, s, torch.randn(n, generator=torch.Generator().manual_seed(5)) * 0.1


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("packed", [False, True])
def test_output_forms_same_bits(m, n, half, packed):
    """Rows of 16-byte stores through LDS (a ragged last chunk included), an odd row stride, a misaligned buffer: the
    same bits, only inside [M, N]."""
    x, w, s, b = _operands(m, n)
    rows = torch.tensor([0, 1, 255, 256, m // 2, m - 2, m - 1])
    ref = block_fp8.reference(x[rows], w, s, native_half=half, bias=b)
    weight = ops.pack_weight(w.cuda()) if packed else w.cuda()
    first = None
    for ld, off in ((n + (-n) % 8 + 8, 0), (n + 4 + (n % 2 == 0), 0), (n + (-n) % 8 + 8, 1)):
        buf = torch.full(((m + 2) * (ld + 8),), SENTINEL, dtype=torch.int16, device="cuda")
        view = buf[off: off + m * ld].view(m, ld)
        ops.block_fp8_gemm(x.cuda(), weight, s.cuda(), b.cuda(), native_half=half, out=view.view(torch.bfloat16)[:, :n])
        got = view[:, :n].clone()
        view[:, :n] = SENTINEL
        assert bool((buf == SENTINEL).all()), f"ld={ld} off={off}: a write outside [M, N]"
        if first is None:
            first = got
            y = got.view(torch.bfloat16)[rows.cuda()].cpu()
            max_rel, mean_rel = block_fp8.parity(y, ref)
            assert max_rel <= block_fp8.MAX_REL_TOL and mean_rel <= block_fp8.MEAN_REL_TOL
        assert torch.equal(got, first)


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("packed", [False, True])
def test_partials_accumulate_to_one_call_bits(m, n, half, packed):
    """Three K ranges added into one fp32 partial, in rows that take 16-byte stores and in rows that do not."""
    x, w, s, b = (t.cuda() for t in _operands(m, n))
    weight = ops.pack_weight(w) if packed else w
    one = ops.block_fp8_gemm(x, weight, s, b, native_half=half)
    for ld in (n + (-n) % 4, n + 2):
        buf = torch.full((m, ld), 7.0, dtype=torch.float32, device="cuda")
        for i, (off, length) in enumerate(RANGES):
            ops.block_fp8_gemm_kslice(x, weight, s, off, length, native_half=half, out=buf[:, :n], accumulate=i > 0)
        assert bool((buf[:, n:] == 7.0).all())
        assert torch.equal(ops.partial_finish(buf[:, :n], b).view(torch.int16), one.view(torch.int16))
