"""Device products with a short inner dimension and a C of many tiles (tmm_device_gemm): these run on one of three
kernels by the cost of a tile's first loads and of its C. Integer data, so the result must be exact; C
holds NaN where beta is 0, and the padding rows of A and B hold NaN."""
import numpy as np
import pytest

import oracle
import tiledmm
from helpers import int_matrix
from test_gpu_ragged import CODES, _ops

pytestmark = pytest.mark.gpu


# one k, whole and partial k-steps, both sides of each type's longest short one; sizes of less than one 128 x 128 tile per
# CU, one, and several
@pytest.mark.parametrize("k", [1, 8, 33, 64, 128, 129, 160, 161, 256, 257, 512, 513])
@pytest.mark.parametrize("m,n", [(897, 705), (2001, 1999), (3003, 2817)])
@pytest.mark.parametrize("dtype", list(CODES), ids=["s", "d", "c", "z"])
def test_short_inner_dimension_exact(torch_gpu, dtype, m, n, k):
    torch = torch_gpu
    cplx = np.issubdtype(dtype, np.complexfloating)
    rng = np.random.default_rng(m + k)
    op = {"N": lambda x: x, "T": lambda x: x.T, "C": lambda x: x.conj().T}
    wide = np.complex128 if cplx else np.float64
    with tiledmm.Handle(CODES[dtype], 1) as h:
        for i, (ta, tb) in enumerate(_ops(dtype)):
            if (i + k) % 2 and m * n > 897 * 705:  # half of the combinations at a time for the large ones
                continue
            ar, ac = oracle.op_shape(ta, m, k)
            br, bc = oracle.op_shape(tb, k, n)
            pad = i % 2
            a, b = int_matrix(rng, ar, ac, dtype, ld=ar + pad), int_matrix(rng, br, bc, dtype, ld=br + pad)
            a[ar:], b[br:] = np.nan, np.nan
            da, db = (torch.from_numpy(np.ascontiguousarray(x.reshape(-1, order="F"))).cuda() for x in (a, b))
            prod = torch.from_numpy(op[ta](a[:ar].astype(wide))).cuda() @ torch.from_numpy(op[tb](b[:br].astype(wide)).copy()).cuda()
            for beta in (0.0, 3.0):
                c = int_matrix(rng, m, n, dtype)
                ref = 2.0 * prod + (beta * torch.from_numpy(c.astype(wide)).cuda() if beta else 0)
                if not beta:
                    c[:] = np.nan
                dc = torch.from_numpy(np.ascontiguousarray(c.reshape(-1, order="F"))).cuda()
                h.device_gemm(ta, tb, m, n, k, 2.0, da, ar + pad, db, br + pad, beta, dc, m)
                h.synchronize()
                out = dc.view(n, m).T.to(ref.dtype)
                assert torch.equal(out, ref), f"{ta}{tb} {m}x{n}x{k} beta {beta} pad {pad}"
