"""The finite-input check at the edges of its vector loads: one bad value anywhere is found, none is not."""

import pytest
import torch

from gaudi_kernels import ops

pytestmark = pytest.mark.gpu


def _case(n, k, m, offset, stride):
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    wbuf = torch.randint(0, 127, (n * k + 16,), dtype=torch.uint8, device="cuda", generator=gen)
    xbuf = torch.randn(m * stride + 8, device="cuda", generator=gen).bfloat16()
    w = wbuf[offset:offset + n * k].view(n, k)
    x = xbuf[offset:offset + m * stride].view(m, stride)[:, :k]
    return x, w, torch.rand((n + 127) // 128, (k + 127) // 128, device="cuda", generator=gen)


# small and odd; row-strided x; misaligned buffers; past the unrolled loads of 1024 workgroups (16 MB of codes)
@pytest.mark.parametrize("n,k,m,offset,pad", [(1, 1, 1, 0, 0), (3, 37, 5, 0, 0), (64, 256, 3, 0, 8), (33, 129, 4, 1, 0),
                                              (4099, 4100, 1030, 0, 0)])
def test_inputs_finite(n, k, m, offset, pad):
    x, w, s = _case(n, k, m, offset, k + pad)
    assert ops.inputs_finite(x, w, s)
    for t, bads in ((x, (float("inf"), float("-inf"), float("nan"))), (w, (0x7F, 0xFF)),
                    (s, (float("inf"), float("nan"), -1.0))):
        last = (t.shape[0] - 1, t.shape[1] - 1)
        for at in {(0, 0), last, (t.shape[0] // 2, t.shape[1] // 3), (last[0], 0), (0, last[1])}:
            for bad in bads:
                kept = t[at].clone()
                t[at] = bad
                assert not ops.inputs_finite(x, w, s)
                t[at] = kept
    # the largest finite values and the codes beside NaN pass
    x[0, 0], w[0, 0], s[0, 0] = torch.finfo(torch.bfloat16).max, 0xFE, torch.finfo(torch.float32).max
    assert ops.inputs_finite(x, w, s)
