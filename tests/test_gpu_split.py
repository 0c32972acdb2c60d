"""Device products with a small C and a long inner dimension (tmm_device_gemm), whose tiles several
workgroups share. Integer data, so the result must be exact whatever the order of the sums."""
import threading

import numpy as np
import pytest

import tiledmm
from test_gpu_ragged import _exact, _ops

pytestmark = pytest.mark.gpu

# one element; one tile; ragged edges of every tile shape; odd inner dimensions and paddings
SHAPES = [(1, 1, 9001, 0), (16, 16, 4104, 1), (17, 33, 7011, 3), (49, 48, 8193, 0), (100, 100, 5999, 2), (129, 65, 6000, 1),
          (300, 420, 8013, 0)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
@pytest.mark.parametrize("m,n,k,pad", SHAPES)
def test_split_exact(torch_gpu, dtype, m, n, k, pad):
    _exact(torch_gpu, dtype, m, n, k, _ops(dtype), pad)


def _problem(torch, m, n, k, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randint(-9, 10, (m, k), generator=gen, device="cuda").double()  # A^T: column-major k x m
    b = torch.randint(-9, 10, (n, k), generator=gen, device="cuda").double()
    return a, b, torch.zeros(n, m, dtype=torch.float64, device="cuda"), (b.cpu() @ a.cpu().T).numpy()


def _call(h, p, stream):
    a, b, c, _ = p
    (m, k), n = a.shape, b.shape[0]
    h.device_gemm("T", "N", m, n, k, 1.0, a, k, b, k, 0.0, c, m, stream=stream.cuda_stream)


def test_split_streams_and_threads(torch_gpu):
    """One handle, two threads with a stream each: their products share the buffer of partial sums."""
    torch = torch_gpu
    sets = [[_problem(torch, *size, seed=10 * t + i) for i, size in enumerate(((64, 64, 30000), (200, 300, 9000), (20, 500, 12000)))]
            for t in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    errors = []

    def work(t):
        try:
            for i in range(30):
                _call(h, sets[t][i % 3], streams[t])
        except Exception as e:  # shown in the main thread
            errors.append(e)

    with tiledmm.Handle(tiledmm.F64, 1) as h:
        threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
    assert not errors, errors
    for p in sets[0] + sets[1]:
        np.testing.assert_array_equal(p[2].cpu().numpy(), p[3])


def test_split_beside_a_graph(torch_gpu):
    """A captured call keeps off the buffer: replays run between and beside calls that use it."""
    torch = torch_gpu
    one, two = _problem(torch, 64, 96, 20000, 1), _problem(torch, 80, 50, 25000, 2)
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    with tiledmm.Handle(tiledmm.F64, 1) as h:
        _call(h, two, other)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            _call(h, one, side)
        for _ in range(3):
            one[2].zero_()
            two[2].zero_()
            torch.cuda.synchronize()
            graph.replay()
            _call(h, two, other)
            torch.cuda.synchronize()
            np.testing.assert_array_equal(one[2].cpu().numpy(), one[3])
            np.testing.assert_array_equal(two[2].cpu().numpy(), two[3])
