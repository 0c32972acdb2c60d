"""The largest complex double device products, whose kernel depends on the layout of the operands. Every row of op(A)
and every column of op(B) is constant, with small integers, so that C is known exactly."""
import pytest

import tiledmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", ["NN", "TT", "CN"])
def test_large_zgemm_exact(torch_gpu, flags):
    torch = torch_gpu
    m, n, k = 23999, 24001, 10601
    u = torch.complex((torch.arange(m, device="cuda") % 7 - 3).double(), (torch.arange(m, device="cuda") % 3).double())
    v = torch.complex((torch.arange(n, device="cuda") % 5).double(), (torch.arange(n, device="cuda") % 4 - 1).double())
    # column-major storage is the transposed tensor
    a = u[None, :].expand(k, m) if flags[0] == "N" else (u.conj() if flags[0] == "C" else u)[:, None].expand(m, k)
    b = v[:, None].expand(n, k) if flags[1] == "N" else v[None, :].expand(k, n)
    a, b = a.contiguous().resolve_conj(), b.contiguous()
    c = torch.empty(n, m, dtype=torch.complex128, device="cuda")
    torch.cuda.synchronize()  # the handle's stream does not wait for torch's
    with tiledmm.Handle(tiledmm.C64, 1) as h:
        h.device_gemm(flags[0], flags[1], m, n, k, 1.0, a, a.shape[1], b, b.shape[1], 0.0, c, m)
        h.synchronize()
    for j in range(0, n, 4000):
        assert torch.equal(c[j:j + 4000], v[j:j + 4000, None] * u[None, :] * k)
