"""The status read-back of the codec and the input check from several threads and streams at once."""

import threading

import pytest
import torch

from gaudi_kernels import _native as nat
from gaudi_kernels import ops

pytestmark = pytest.mark.gpu


def test_threads_and_streams():
    codes = [torch.full((512 + 16 * t,), 1, dtype=torch.uint8, device="cuda") for t in range(4)]  # every code rounds
    bad = torch.tensor([0x7F] * 512, dtype=torch.uint8, device="cuda")
    scales = torch.ones(4, device="cuda")
    torch.cuda.synchronize()
    wrong = []

    def work(t):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                if ops.codec_ocp_to_half(codes[t], scales)[2] != codes[t].numel():
                    wrong.append(t)
                try:
                    ops.codec_ocp_to_half(bad, scales)
                    wrong.append(t)
                except nat.GkError as e:
                    if e.status != nat.GK_NONFINITE_CODE:
                        wrong.append(e.status)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not wrong


def test_stream_handle_is_the_current_stream():
    device = torch.device("cuda", torch.cuda.current_device())
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            assert ops._stream(device) == stream.cuda_stream
