"""The wrappers launch on the calling thread's current stream of the tensors' device."""

import threading

import pytest
import torch

from kernels._hip import stream
from kernels.dequant_matmul import int8_matmul
from serve.quantize import quantize_int8

pytestmark = pytest.mark.gpu


def _handle(dev):
    return torch.cuda.current_stream(dev).cuda_stream


def test_current_stream_of_the_thread():
    dev = torch.zeros(1, device="cuda").device
    side, seen = torch.cuda.Stream(), {}

    def other():
        seen["other"] = (stream(dev), _handle(dev))

    assert stream(dev) == _handle(dev)
    with torch.cuda.stream(side):
        assert stream(dev) == _handle(dev) == side.cuda_stream
        t = threading.Thread(target=other)
        t.start()
        t.join()
    assert seen["other"][0] == seen["other"][1] != side.cuda_stream


def test_capture_and_replay():
    g = torch.Generator(device="cuda").manual_seed(0)
    w_q, s = quantize_int8(torch.randn(96, 256, generator=g, device="cuda"))
    x = torch.randn(8, 256, generator=g, device="cuda")
    want = int8_matmul(x, w_q, s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert stream(x.device) == _handle(x.device)
        y = int8_matmul(x, w_q, s)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
