"""Which operands the direct FP32 kernels take: a load's 32-bit offsets have to reach every row of
A and B that one load spans. The library's own rule, asked on the host."""
import ctypes

import pytest

from conftest import phpc


class F32Desc(ctypes.Structure):
    _fields_ = [("A", ctypes.c_void_p), ("B", ctypes.c_void_p), ("C", ctypes.c_void_p),
                ("lda", ctypes.c_long), ("ldb", ctypes.c_long), ("ldc", ctypes.c_long),
                ("m", ctypes.c_int), ("n", ctypes.c_int), ("k", ctypes.c_int),
                ("tiles_n", ctypes.c_int), ("tile_start", ctypes.c_int)]


def direct_ok(lib, m, k, n, lda, ldb):
    fn = lib["_Z18phpc_f32_direct_okPK7F32Desci"]
    fn.restype, fn.argtypes = ctypes.c_bool, [ctypes.POINTER(F32Desc), ctypes.c_int]
    return fn(ctypes.byref(F32Desc(lda=lda, ldb=ldb, ldc=n, m=m, n=n, k=k)), 1)


FIRST_TOO_LONG = 2 ** 31 // 32  # eight rows of so many floats span 2 GiB


@pytest.mark.parametrize("m", [1, 3, 5000])
@pytest.mark.parametrize("k", [FIRST_TOO_LONG, 153391690, 160000000, 2 ** 29, 2 ** 30, 2 ** 31 - 1])
def test_rows_of_a_too_long(lib, m, k):
    assert not direct_ok(lib, m, k, 1, k, 1)


@pytest.mark.parametrize("m,k,lda", [(1, FIRST_TOO_LONG - 1, FIRST_TOO_LONG - 1), (4, 37, 2 ** 40), (300, 4096, 4096),
                                     (2, FIRST_TOO_LONG - 1, 2 ** 33)])
def test_rows_of_a_that_fit(lib, m, k, lda):
    assert direct_ok(lib, m, k, 1, lda, 1)


@pytest.mark.gpu
def test_rows_too_long_are_refused():
    import torch
    k = FIRST_TOO_LONG
    A, B = torch.zeros(1, k, device="cuda"), torch.zeros(k, 1, device="cuda")
    C = torch.zeros(1, 1, device="cuda")
    with pytest.raises(RuntimeError, match="leading dimension too large"):
        phpc.sgemm_device(A, B, C, method=phpc.SGEMM_FP32)
    plan = phpc.Plan(phpc.F32, [(A, B, C)])
    with pytest.raises(RuntimeError, match="leading dimension too large"):
        plan.launch()
    plan.close()
