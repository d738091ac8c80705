"""Host matrices through the pinned slots: pieces, parts and lanes at their edges. k = 1, so that
every output is exactly c + a b."""
import numpy as np
import pytest

from conftest import phpc

pytestmark = pytest.mark.gpu


# one piece in all; several 2 MiB pieces with a ragged last one; rows longer than a piece; 64 MiB
# and more, where pieces grow; more pieces than slots (4 buffers of 32 MiB)
@pytest.mark.parametrize("m,n", [(1, 1), (300, 500), (513, 511), (1025, 1300), (3, 300001), (2900, 3001), (5200, 4099)])
def test_pieces(m, n):
    rng = np.random.default_rng(m + n)
    a, b = rng.uniform(-1, 1, (m, 1)), rng.uniform(-1, 1, (1, n))
    c = rng.uniform(-1, 1, (m, n))
    want = c + a * b
    for _ in range(2):  # slots of another size in between
        got = c.copy()
        phpc.gemm_cuda(a, b, got)
        assert np.array_equal(got, want)
        small = np.ones((2, 2))
        phpc.gemm_cuda(np.ones((2, 1)), np.ones((1, 2)), small)
        assert np.all(small == 2.0)


def test_strided_rows():
    rng = np.random.default_rng(4)
    a, b = rng.uniform(-1, 1, (900, 1)), rng.uniform(-1, 1, (1, 700))
    buf = rng.uniform(-1, 1, (900, 733))
    want = buf.copy()
    want[:, :700] += a * b
    phpc.gemm_cuda(a, b, buf, n=700, ldc=733)
    assert np.array_equal(buf, want)
