"""Emulated DGEMM with so many rows that the workgroups of their exponents exceed one dimension of a grid (2^32 threads,
1024 for 16 rows). Integer data: exact."""
import pytest

import tiledmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("option,value", [(tiledmm.OPT_OZAKI_MODULI, 8), (tiledmm.OPT_OZAKI_SLICES, 4)])
def test_emulation_of_many_rows(torch_gpu, option, value):
    torch = torch_gpu
    m, n, k = (1 << 26) + 5, 3, 2
    a = torch.arange(m * k, device="cuda").remainder_(7).sub_(3).double().view(k, m)  # column-major m x k
    a[1, -1] = 1000.0  # the last row's exponent differs from the others'
    b = torch.tensor([[1.0, -2.0], [3.0, 5.0], [0.0, 700.0]], dtype=torch.float64, device="cuda")  # column-major k x n
    c = torch.full((n, m), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    with tiledmm.Handle(tiledmm.F64, 1) as h:
        h.set_option(option, value)
        h.device_gemm("N", "N", m, n, k, 1.0, a, m, b, k, 0.0, c, m)
        h.synchronize()
    for j in range(n):
        assert torch.equal(c[j], b[j, 0] * a[0] + b[j, 1] * a[1]), f"column {j}"
    del a, b, c
    torch.cuda.empty_cache()
