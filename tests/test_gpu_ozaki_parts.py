"""Emulated DGEMM (Ozaki scheme II) around the operand sizes from which one set of workgroups writes the
residues of all moduli. Integer data: exact."""
import numpy as np
import pytest

import tiledmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("moduli", [6, 13, 16, 20])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (700, 650, 700), (768, 768, 1024), (769, 768, 1025), (65, 3000, 63)])
def test_residues_of_small_operands(torch_gpu, m, n, k, moduli):
    torch = torch_gpu
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-3, 4, (m, k), generator=gen, device="cuda").double()  # A^T: column-major k x m
    b = torch.randint(-3, 4, (n, k), generator=gen, device="cuda").double()
    c = torch.full((n, m), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    with tiledmm.Handle(tiledmm.F64, 1) as h:
        h.set_option(tiledmm.OPT_OZAKI_MODULI, moduli)
        h.device_gemm("T", "N", m, n, k, 1.0, a, k, b, k, 0.0, c, m)
        h.synchronize()
    np.testing.assert_array_equal(c.cpu().numpy(), b.cpu().numpy() @ a.cpu().numpy().T)
