"""The CRT split GEMM's residue products at the edges of their tiles, row blocks and slabs: on
integer operands the result is the exact integer product, whatever the tile, with everything
around C untouched."""
import numpy as np
import pytest

from conftest import phpc

pytestmark = pytest.mark.gpu


def run(m, k, n, lim, moduli=0):
    import torch
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    A = rng.integers(-lim, lim + 1, (m, k))
    B = rng.integers(-lim, lim + 1, (k, n))
    buf = torch.full((m + 2, n + 3), 7.0, dtype=torch.float64, device="cuda")
    C = buf[1:1 + m, 1:1 + n]
    C.zero_()
    phpc.dgemm_split_device(torch.from_numpy(A.astype(np.float64)).cuda(), torch.from_numpy(B.astype(np.float64)).cuda(),
                            C, slices=moduli, method=phpc.SPLIT_CRT)
    torch.cuda.synchronize()
    assert np.array_equal(C.cpu().numpy(), (A @ B).astype(np.float64)), (m, k, n)
    C.fill_(7.0)
    assert torch.all(buf == 7.0)


# row blocks of 16, slabs of 64 k (kp a multiple of 128), a ring of three or four slabs and steady
# turns of four or six; 64x64 tiles (few), 128x128 and 256x256 ones (many)
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (15, 63, 17), (16, 64, 16), (17, 65, 15), (63, 128, 65), (65, 129, 63),
                                   (33, 257, 130), (64, 700, 64), (1, 900, 300), (300, 900, 1), (1000, 200, 1003),
                                   (1025, 511, 1279), (2300, 640, 2305), (2305, 130, 2600)])
def test_edges_exact(m, k, n):
    run(m, k, n, 1 << 18)


def test_each_tile_with_many_moduli():
    run(130, 300, 260, 1 << 20, 20)
    run(1500, 300, 1300, 1 << 20, 20)
    run(2400, 300, 2100, 1 << 20, 20)


@pytest.mark.parametrize("k", [130944, 130945, 262000])
def test_sums_longer_than_one_piece(k):
    """k past 130944 residue products, the most that an int32 holds: reduced in between."""
    run(20, k, 35, 100)
