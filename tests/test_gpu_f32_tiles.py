"""FP32 direct-to-LDS kernels at the edges of their tiles, slabs and tails: the bits of the
register-staged kernels (one FMA chain per output in k order) on operands whose rows start at odd
offsets with odd strides, with everything around C untouched."""
import pytest

from conftest import phpc

pytestmark = pytest.mark.gpu


def on_view(x, fill):
    """x as a view at an odd offset of a buffer with an odd row stride."""
    import torch
    m, n = x.shape
    buf = torch.full((m + 2, n + 5 - n % 2), fill, dtype=torch.float32, device="cuda")
    v = buf[1:1 + m, 1:1 + n]
    v.copy_(x)
    return buf, v


def inputs(m, k, n, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return tuple(torch.empty(s, device="cuda").uniform_(-1, 1, generator=g) for s in ((m, k), (k, n), (m, n)))


def staged(A, B, C0):
    """C0 + A B on the register-staged kernels, contiguous operands."""
    import torch
    C = C0.clone()
    phpc.set_tuning(phpc.TUNE_F32_TRANSPOSED_A, 0)
    try:
        phpc.sgemm_device(A, B, C, method=phpc.SGEMM_FP32)
        torch.cuda.synchronize()
    finally:
        phpc.set_tuning(phpc.TUNE_F32_TRANSPOSED_A, 1)
    return C


# k around whole slabs (32 or 64 deep) and the ring's depth of slabs, m and n one off the tiles'
# edges; then sizes on 64x64 tiles with a 32x32 tail (by rows, by columns) and on 128x64 tiles
# with a 64x64 tail, on 256 CUs
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (31, 31, 33), (65, 33, 63), (129, 64, 127), (255, 65, 257),
                                   (33, 97, 31), (64, 160, 129), (40, 401, 31), (1, 300, 700), (700, 300, 1),
                                   (1100, 35, 1001), (500, 40, 2301), (1100, 161, 1001), (4100, 20, 2201), (1023, 63, 1000), (961, 257, 1024),
                                   (2200, 67, 4301), (4096, 129, 2049)])
def test_tile_slab_and_tail_edges(m, k, n):
    import torch
    A, B, C0 = inputs(m, k, n, 7 * m + 3 * k + n)
    # what surrounds the operands is NaN: an entry of padding that reached an output would show
    _, dA = on_view(A, float("nan"))
    _, dB = on_view(B, float("nan"))
    buf, dC = on_view(C0, 7.0)
    phpc.sgemm_device(dA, dB, dC, method=phpc.SGEMM_FP32)
    torch.cuda.synchronize()
    assert torch.equal(dC, staged(A, B, C0)), (m, k, n)
    want = (C0.double() + A.double() @ B.double()).float()
    bound = (k + 2) * 2.0 ** -23 * (C0.abs() + A.abs() @ B.abs())
    assert torch.all((dC - want).abs() <= bound)
    dC.fill_(7.0)
    assert torch.all(buf == 7.0)


def test_special_values():
    """Infinities, NaNs, subnormals and signed zeros go through the chain as FMAs do."""
    import torch
    A, B, C0 = inputs(130, 70, 90, 5)
    A[3, 4], A[9, 60], B[7, 11], B[69, 89] = float("inf"), float("nan"), float("-inf"), 1e-40
    A[20, :], C0[20, :] = -0.0, -0.0
    C = C0.clone()
    phpc.sgemm_device(A, B, C, method=phpc.SGEMM_FP32)
    want = staged(A, B, C0)
    assert torch.equal(C.isnan(), want.isnan())
    fin = ~want.isnan()
    assert torch.equal(C.view(torch.int32)[fin], want.view(torch.int32)[fin])


# many GEMMs as one plan, so the descriptors go through the device list and its index (an entry
# for every 64 tiles): more GEMMs than tiles per entry, several entries within one GEMM, one
# without work between, and a tail
@pytest.mark.parametrize("shapes", [
    [(i % 7 + 1, 5 + i % 3, i % 5 + 1) for i in range(150)],
    [(33, 40, 31), (1500, 40, 1500), (8, 9, 0), (64, 64, 64)],
    [(900, 64, 700), (400, 48, 333), (300, 33, 255)],
    [(4100, 33, 4101), (130, 64, 70), (2100, 32, 1025), (31, 65, 1000)],
])
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_many_gemms_as_one_plan(shapes, dtype):
    import torch
    f64 = dtype == "f64"
    items = [inputs(*s, seed=i) for i, s in enumerate(shapes)]
    if f64:
        items = [tuple(x.double() for x in it) for it in items]
    want = []
    for A, B, C0 in items:
        C = C0.clone()
        if C.numel():
            if f64:
                phpc.dgemm_device(A, B, C)
            else:
                C = staged(A, B, C0)
        want.append(C)
    plan = phpc.Plan(phpc.F64 if f64 else phpc.F32, items)
    plan.launch()
    torch.cuda.synchronize()
    for (_, _, C), w in zip(items, want):
        assert torch.equal(C, w)
    plan.close()


# rows of B shorter than a 16-byte load, B ending where its rows end: the last slab, or the last two,
# hold rows whose loads would reach past it
@pytest.mark.parametrize("k", [33, 34, 35, 65, 66, 97, 129, 161, 290])
@pytest.mark.parametrize("m,n", [(1, 1), (40, 1), (5, 2), (300, 3), (2000, 1), (70000, 1)])
def test_short_rows_of_b(m, n, k):
    import torch
    A, B, C0 = inputs(m, k, n, 11 * m + k + n)
    C = C0.clone()
    phpc.sgemm_device(A, B, C, method=phpc.SGEMM_FP32)
    torch.cuda.synchronize()
    assert torch.equal(C, staged(A, B, C0)), (m, k, n)
    if n == 1:  # a column of rows of two: ldb = 2
        wide = torch.stack([B[:, 0], torch.full_like(B[:, 0], float("nan"))], dim=1)
        D = C0.clone()
        phpc.sgemm_device(A, wide[:, :1], D, method=phpc.SGEMM_FP32)
        torch.cuda.synchronize()
        assert torch.equal(D, C), (m, k, n)


# beside the lines of the tile rule below one 64x64 tile per CU (256): k, and the tiles
@pytest.mark.parametrize("m,k,n", [(1023, 999, 1000), (1023, 1000, 1000), (961, 1027, 1024), (800, 1000, 960),
                                   (769, 1065, 1023), (1025, 1001, 1023)])
def test_about_one_tile_per_cu(m, k, n):
    import torch
    A, B, C0 = inputs(m, k, n, m + k)
    _, dA = on_view(A, float("nan"))
    _, dB = on_view(B, float("nan"))
    C = C0.clone()
    phpc.sgemm_device(dA, dB, C, method=phpc.SGEMM_FP32)
    torch.cuda.synchronize()
    assert torch.equal(C, staged(A, B, C0))
    x, y, z = (t.double() for t in (A, B, C0))
    want = z.clone()
    phpc.dgemm_device(x, y, z)
    phpc.set_launch_policy(0, 2, 0)  # register-staged
    try:
        phpc.dgemm_device(x, y, want)
        torch.cuda.synchronize()
    finally:
        phpc.set_launch_policy(0, -1, 0)
    assert torch.equal(z, want)
