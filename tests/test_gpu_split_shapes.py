"""Every tile shape of the kernels that share a product's tiles among workgroups (tmm_device_gemm, small C and long
inner dimension), of every element type and in all op combinations, at odd sizes and at whole tiles. The
handle has to report that shape for the call; integer data, so the result must be exact."""
import numpy as np
import pytest

import tiledmm
from test_gpu_ragged import _exact, _ops

pytestmark = pytest.mark.gpu

D, S, Z, C = np.float64, np.float32, np.complex128, np.complex64


@pytest.mark.parametrize("dtype,edge,m,n,k", [
    (D, 16, 17, 33, 3001), (D, 16, 32, 16, 4096), (D, 32, 115, 135, 4003), (D, 32, 96, 128, 4096),
    (D, 48, 137, 475, 4501), (D, 48, 144, 240, 6400), (D, 64, 441, 297, 4507), (D, 64, 320, 448, 4800),
    (S, 16, 17, 33, 9001), (S, 16, 32, 16, 8192), (S, 32, 99, 113, 7001), (S, 32, 96, 160, 6400),
    (S, 48, 277, 141, 8003), (S, 48, 192, 240, 8000), (S, 64, 571, 251, 6005), (S, 64, 448, 320, 6400),
    (Z, 16, 17, 33, 1501), (Z, 16, 32, 16, 2048), (Z, 32, 213, 113, 2501), (Z, 32, 320, 448, 1280),
    (Z, 48, 355, 357, 1501), (Z, 48, 384, 384, 1504),
    (C, 16, 17, 33, 2501), (C, 16, 32, 16, 3200), (C, 32, 99, 163, 3001), (C, 32, 128, 160, 2608),
    (C, 48, 351, 369, 2001), (C, 48, 384, 384, 2048),
])
def test_split_shapes_exact(torch_gpu, monkeypatch, dtype, edge, m, n, k):
    if torch_gpu.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are chosen for 256 CUs")
    splits = []

    class Recording(tiledmm.Handle):
        def device_gemm(self, *args, **kwargs):
            super().device_gemm(*args, **kwargs)
            splits.append(self.last_device_split())

    monkeypatch.setattr(tiledmm, "Handle", Recording)
    _exact(torch_gpu, dtype, m, n, k, _ops(dtype), 1 if m % 2 else 0)
    assert len(splits) == len(_ops(dtype)) and all(e == edge and parts > 1 for e, parts in splits), splits


def test_products_that_are_not_split(torch_gpu):
    """A short inner dimension, and alpha = 0 (nothing to add up)."""
    torch = torch_gpu
    a, b, c = (torch.zeros(64 * 9000, dtype=torch.float64, device="cuda") for _ in range(3))
    with tiledmm.Handle(tiledmm.F64, 1) as h:
        h.device_gemm("T", "N", 64, 64, 9000, 1.0, a, 9000, b, 9000, 0.0, c, 64)
        assert h.last_device_split()[1] > 1
        h.device_gemm("T", "N", 64, 64, 100, 1.0, a, 100, b, 100, 0.0, c, 64)
        assert h.last_device_split() == (0, 1)
        h.device_gemm("T", "N", 64, 64, 9000, 1.0, a, 9000, b, 9000, 0.0, c, 64)
        h.device_gemm("T", "N", 64, 64, 9000, 0.0, a, 9000, b, 9000, 0.0, c, 64)
        assert h.last_device_split() == (0, 1)
        h.synchronize()
