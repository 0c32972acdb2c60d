"""Device products whose C has more small tiles than a launch takes (2^32 threads in a grid, 256 per tile): the kernels of
larger tiles run them. op(A) and op(B) hold small integers, so that C is known exactly."""
import pytest

import tiledmm

pytestmark = pytest.mark.gpu


# 2^24 tiles of 32 x 32 with a C that is read; of 32 x 16; of 32 x 32 with a C of NaN
@pytest.mark.parametrize("code,name,m,n,k,flags,beta", [
    (tiledmm.F32, "float32", 131072, 131072, 2, "NT", 1.0),
    (tiledmm.C64, "complex128", 1 << 29, 1, 1, "TN", 0.0),
    (tiledmm.F64, "float64", (1 << 29) + 1, 17, 1, "TN", 0.0),
])
def test_more_tiles_than_a_grid_exact(torch_gpu, code, name, m, n, k, flags, beta):
    torch = torch_gpu
    dtype = getattr(torch, name)

    def ints(rows, cols, mod):  # small integers, exact in every type
        x = torch.arange(rows * cols, device="cuda").remainder_(mod).sub_(mod // 2).to(dtype)
        return x.view(rows, cols)

    a, b = ints(m, k, 7), ints(k, n, 5)  # op(A), op(B); column-major storage is the transposed tensor
    da = a.t().contiguous() if flags[0] == "N" else a
    db = b.t().contiguous() if flags[1] == "N" else b
    c = torch.full((n, m), 3.0 if beta else float("nan"), dtype=dtype, device="cuda")
    torch.cuda.synchronize()  # the handle's stream does not wait for torch's
    with tiledmm.Handle(code, 1) as h:
        h.device_gemm(flags[0], flags[1], m, n, k, 1.0, da, da.shape[1], db, db.shape[1], beta, c, m)
        h.synchronize()
    step = max(1, (1 << 30) // m)
    for j in range(0, n, step):
        want = torch.full((min(step, n - j), m), 3.0 if beta else 0.0, dtype=dtype, device="cuda")
        for x in range(k):
            want += b[x, j:j + step, None] * a[None, :, x]
        assert torch.equal(c[j:j + step], want), f"columns {j}"
    del a, b, c, da, db, want
    torch.cuda.empty_cache()
