"""Device products of ragged shapes (tmm_device_gemm): inner dimensions that are no whole number of
k-steps and row counts that are no whole number of 16-byte chunks, for every element type and op
combination. Integer data, so the result must be exact; the padding rows of A and B hold NaN, so a
value read from outside a matrix shows in C."""
import numpy as np
import pytest

import oracle
import tiledmm
from helpers import int_matrix

pytestmark = pytest.mark.gpu

CODES = {np.float32: tiledmm.F32, np.float64: tiledmm.F64, np.complex64: tiledmm.C32, np.complex128: tiledmm.C64}


def _exact(torch, dtype, m, n, k, ops, pad):
    cplx = np.issubdtype(dtype, np.complexfloating)
    alpha, beta = (2 - 1j, 1 + 3j) if cplx else (2.0, 3.0)
    wide = np.complex128 if cplx else np.float64
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    with tiledmm.Handle(CODES[dtype], 1) as h:
        for ta, tb in ops:
            ar, ac = oracle.op_shape(ta, m, k)
            br, bc = oracle.op_shape(tb, k, n)
            A, B = int_matrix(rng, ar, ac, dtype, ld=ar + pad), int_matrix(rng, br, bc, dtype, ld=br + pad)
            A[ar:], B[br:] = np.nan, np.nan
            C = int_matrix(rng, m, n, dtype)
            op = {"N": lambda X: X, "T": lambda X: X.T, "C": lambda X: X.conj().T}
            ref = alpha * (op[ta](A[:ar].astype(wide)) @ op[tb](B[:br].astype(wide))) + beta * C.astype(wide)
            dA, dB, dC = (torch.from_numpy(np.ascontiguousarray(X.reshape(-1, order="F"))).cuda() for X in (A, B, C))
            h.device_gemm(ta, tb, m, n, k, alpha, dA, ar + pad, dB, br + pad, beta, dC, m)
            h.synchronize()
            out = dC.cpu().numpy().reshape(C.shape, order="F").astype(wide)
            np.testing.assert_array_equal(out, ref, err_msg=f"{ta}{tb} {m}x{n}x{k} pad {pad}")


def _ops(dtype):
    ops = "NTC" if np.issubdtype(dtype, np.complexfloating) else "NT"
    return [(a, b) for a in ops for b in ops]


@pytest.mark.parametrize("k", [1, 7, 17, 263])
@pytest.mark.parametrize("dtype,m,n", [(np.float64, 2945, 2947), (np.float32, 2945, 2946), (np.complex64, 2945, 2947),
                                       (np.complex128, 1473, 1471)], ids=["d", "s", "c", "z"])
def test_pipelined_kernels_ragged(torch_gpu, dtype, m, n, k):
    """At least two workgroup tiles per CU: the software-pipelined kernels."""
    _exact(torch_gpu, dtype, m, n, k, _ops(dtype), 1)


# each of the tile shapes (16 to 64 rows and columns) is the estimated fastest at one of these sizes
KS_SIZES = [(1, 1, 1), (16, 16, 1), (17, 33, 5), (457, 1266, 6), (298, 397, 430), (1219, 204, 556), (1213, 416, 178),
            (645, 1123, 536), (1186, 631, 381), (476, 1159, 214), (1316, 722, 450), (704, 710, 694), (1059, 1220, 683),
            (1261, 1169, 697), (1302, 1305, 686), (200, 301, 5003)]


@pytest.mark.parametrize("m,n,k", KS_SIZES)
@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex64, np.complex128], ids=["d", "s", "c", "z"])
def test_split_inner_dimension_ragged(torch_gpu, dtype, m, n, k):
    """Fewer tiles: the kernels that split the inner dimension over a workgroup's waves."""
    _exact(torch_gpu, dtype, m, n, k, _ops(dtype), 3 if m > 16 else 2)


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex64, np.complex128], ids=["d", "s", "c", "z"])
def test_leading_dimension_of_one(torch_gpu, dtype):
    """Row vectors without padding: consecutive columns lie one element apart."""
    _exact(torch_gpu, dtype, 1, 1, 100, [("N", "T")], 0)
    _exact(torch_gpu, dtype, 1, 70, 33, [("N", "T"), ("N", "N")], 0)
