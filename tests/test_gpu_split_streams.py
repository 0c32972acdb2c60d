"""Products that several workgroups share (tmm_device_gemm, small C and long inner dimension) on several streams of
one handle: a stream's product does not wait for another stream's, and more streams than the handle keeps buffers for
still get exact results."""
import numpy as np
import pytest

import tiledmm
from test_gpu_split import _call, _problem

pytestmark = pytest.mark.gpu


def _busy(torch, h, stream, a, c, times):
    n = a.shape[0]
    for _ in range(times):
        h.device_gemm("T", "N", n, n, n, 1.0, a, n, a, n, 0.0, c, n, stream=stream.cuda_stream)


def test_streams_do_not_wait_for_each_other(torch_gpu):
    """A stream with some 150 ms of large products before its split one; the other stream's split product,
    issued after it, is done first. Streams may share a hardware queue, so one that a plain kernel can
    use beside the busy stream is looked for."""
    torch = torch_gpu
    one, two = _problem(torch, 64, 96, 20000, 1), _problem(torch, 80, 50, 25000, 2)
    n = 8192
    a, c = torch.ones(n, n, dtype=torch.float64, device="cuda"), torch.empty(n, n, dtype=torch.float64, device="cuda")
    x = torch.zeros(64, device="cuda")
    first = torch.cuda.Stream()
    with tiledmm.Handle(tiledmm.F64, 1) as h, tiledmm.Handle(tiledmm.F64, 1) as large:
        _call(h, one, first)
        torch.cuda.synchronize()
        for _ in range(8):
            second = torch.cuda.Stream()
            done = torch.cuda.Event()
            _busy(torch, large, first, a, c, 4)
            done.record(first)
            with torch.cuda.stream(second):
                x.add_(1)
            second.synchronize()
            beside = not done.query()
            torch.cuda.synchronize()
            if beside:
                break
        else:
            pytest.skip("no stream runs beside the first one")
        before = []
        for _ in range(2):  # the first round also allocates the second stream's buffer
            for p in (one, two):
                p[2].zero_()
            torch.cuda.synchronize()
            done = torch.cuda.Event()
            _busy(torch, large, first, a, c, 10)
            _call(h, one, first)
            done.record(first)
            _call(h, two, second)
            second.synchronize()
            before.append(not done.query())
            torch.cuda.synchronize()
            for p in (one, two):
                np.testing.assert_array_equal(p[2].cpu().numpy(), p[3])
        assert before[1], before


def test_more_streams_than_buffers(torch_gpu):
    torch = torch_gpu
    problems = [_problem(torch, 48 + i, 64, 9000 + 8 * i, i) for i in range(12)]
    streams = [torch.cuda.Stream() for _ in problems]
    torch.cuda.synchronize()
    with tiledmm.Handle(tiledmm.F64, 1) as h:
        for _ in range(10):
            for p, s in zip(problems, streams):
                _call(h, p, s)
        torch.cuda.synchronize()
    for p in problems:
        np.testing.assert_array_equal(p[2].cpu().numpy(), p[3])
