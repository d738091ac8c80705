"""FP64 tile configurations at the edges of their tiles, slabs and tails: bit-exact against the
oracle's restatement of the reference kernel (src/phpc_gemm.cu:25-55), on operands whose rows
start at odd offsets with odd strides, with everything around C untouched."""
import numpy as np
import pytest

from conftest import phpc
import oracle as O

pytestmark = pytest.mark.gpu

# configurations that read A and B where they lie; the ones that also group k in panels
DIRECT = [3, 4, 5, 7, 9, 10, 11, 12, 13, 14, 15, 16]
PANELS = [3, 5, 12, 13, 14, 15, 16]


def bits(x):
    return np.ascontiguousarray(x).view(np.uint64)


def on_view(x, fill):
    """x on the device as a view at an odd offset of a buffer with an odd row stride."""
    import torch
    m, n = x.shape
    buf = torch.full((m + 2, n + 5 - n % 2), fill, dtype=torch.float64, device="cuda")
    v = buf[1:1 + m, 1:1 + n]
    v.copy_(torch.from_numpy(x))
    return buf, v


def run(m, k, n, cfg, panel=0):
    import torch
    A, B, C0 = O.uniform((m, k), 1), O.uniform((k, n), 2), O.uniform((m, n), 3)
    # what surrounds the operands is NaN: an entry of padding that reached an output would show
    _, dA = on_view(A, float("nan"))
    _, dB = on_view(B, float("nan"))
    buf, dC = on_view(C0, 7.0)
    phpc.set_launch_policy(0, cfg, 0)
    try:
        phpc.dgemm_device(dA, dB, dC, panel=panel)
        torch.cuda.synchronize()
    finally:
        phpc.set_launch_policy(0, -1, 0)
    want = panel_sums(A, B, C0, panel) if panel else O.kernel_emul(A, B, C0.copy())
    got = buf.cpu().numpy()
    assert np.array_equal(bits(got[1:1 + m, 1:1 + n]), bits(want)), (m, k, n, cfg, panel)
    got[1:1 + m, 1:1 + n] = 7.0
    assert np.all(got == 7.0)


def panel_sums(A, B, C0, panel):
    want = C0.copy()
    for k0 in range(0, A.shape[1], panel):
        k1 = min(A.shape[1], k0 + panel)
        want = want + O.kernel_emul(np.ascontiguousarray(A[:, k0:k1]), np.ascontiguousarray(B[k0:k1]),
                                    np.zeros_like(C0))
    return want


# k around whole slabs (16 or 32 deep) and around the ring's depth of slabs; m and n one off
# the tiles' edges, and an odd n whose last 16-byte piece would end past its row
@pytest.mark.parametrize("cfg", DIRECT)
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (31, 15, 33), (65, 16, 63), (129, 32, 127), (255, 33, 257),
                                   (64, 160, 129), (257, 161, 65), (40, 400, 31), (191, 47, 130),
                                   (193, 64, 127), (400, 20, 129)])
def test_tile_and_slab_edges(cfg, m, k, n):
    run(m, k, n, cfg)


@pytest.mark.parametrize("cfg", PANELS)
@pytest.mark.parametrize("m,k,n,panel", [(70, 130, 65, 16), (130, 200, 129, 33), (33, 300, 257, 64), (64, 97, 40, 96), (193, 70, 129, 48),
                                         (385, 33, 127, 16)])
def test_panel_edges(cfg, m, k, n, panel):
    run(m, k, n, cfg, panel)


# work that the planner cuts into head tiles and a tail of smaller ones: by rows, by columns,
# on 64x64, 256x128 and (with panels) 128x128 heads, on 256 CUs
@pytest.mark.parametrize("m,k,n,panel", [(1023, 33, 1000, 0), (961, 130, 1024, 0), (1023, 33, 1000, 9), (1100, 35, 1001, 0), (500, 40, 2301, 0), (1100, 35, 1001, 16),
                                         (4100, 20, 4201, 0), (4200, 20, 4101, 7), (6200, 33, 6301, 16),
                                         (6301, 20, 6200, 7)])
def test_head_and_tail(m, k, n, panel):
    run(m, k, n, -1, panel)


def test_tail_of_several_gemms_as_one_plan():
    """A plan of three GEMMs whose last two are cut: items equal the same products alone."""
    import torch
    shapes = [(900, 64, 700), (400, 48, 333), (300, 33, 255)]
    items, want = [], []
    for i, (m, k, n) in enumerate(shapes):
        A, B, C0 = O.uniform((m, k), 10 + i), O.uniform((k, n), 20 + i), O.uniform((m, n), 30 + i)
        items.append(tuple(torch.from_numpy(x.copy()).cuda() for x in (A, B, C0)))
        want.append(O.kernel_emul(A, B, C0.copy()))
    plan = phpc.Plan(phpc.F64, items)
    plan.launch()
    torch.cuda.synchronize()
    for (_, _, dC), w in zip(items, want):
        assert np.array_equal(bits(dC.cpu().numpy()), bits(w))
    plan.close()


# rows of A so far apart that a load's rows span 2 GiB: products of one row each
@pytest.mark.parametrize("dtype,lda", [("f64", 34_000_000), ("f32", 68_000_000)])
def test_rows_of_a_far_apart(dtype, lda):
    import torch
    f64 = dtype == "f64"
    tdt = torch.float64 if f64 else torch.float32
    m, k, n = 3, 37, 130
    g = torch.Generator(device="cuda").manual_seed(3)
    far = torch.empty((m - 1) * lda + k, dtype=tdt, device="cuda").as_strided((m, k), (lda, 1))
    A, B, C0 = (torch.randint(-8, 9, s, generator=g, device="cuda").to(tdt) for s in ((m, k), (k, n), (m, n)))
    far.copy_(A)
    want = C0 + (A.double() @ B.double()).to(tdt)  # integers: exact in any order
    C, D, E = C0.clone(), C0.clone(), C0.clone()
    if f64:
        phpc.dgemm_device(far, B, C)
    else:
        phpc.sgemm_device(far, B, C, method=phpc.SGEMM_FP32)
    plan = phpc.Plan(phpc.F64 if f64 else phpc.F32, [(far, B, D), (A, B, E)])
    plan.launch()
    torch.cuda.synchronize()
    plan.close()
    assert torch.equal(C, want) and torch.equal(D, want) and torch.equal(E, want)


# a column of so many rows that a workgroup per tile would take 2^32 threads
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_more_tiles_than_one_launch_starts(dtype):
    import torch
    m = 2 ** 30 + 777
    t = torch.float64 if dtype == "f64" else torch.float32
    A, C = torch.empty(m, 1, dtype=t, device="cuda"), torch.ones(m, 1, dtype=t, device="cuda")
    A[:, 0] = torch.arange(m, device="cuda") % 1021
    B = torch.full((1, 1), 3.0, dtype=t, device="cuda")
    if dtype == "f64":
        phpc.dgemm_device(A, B, C)
    else:
        phpc.sgemm_device(A, B, C, method=phpc.SGEMM_FP32)
    torch.cuda.synchronize()
    A.mul_(3.0).add_(1.0)
    assert torch.equal(A, C)


# GEMMs that go through the shared descriptor buffer in eager calls: captured, their launches carry
# them, and replays do not depend on what eager calls put into that buffer meanwhile
@pytest.mark.parametrize("what", ["far_rows", "ranks", "ranks_with_tails"])
def test_captured_lists(what):
    import torch
    g = torch.Generator(device="cuda").manual_seed(4)

    def ints(*s):
        return torch.randint(-8, 9, s, generator=g, device="cuda").double()

    if what == "far_rows":
        m, k, n, lda = 5, 37, 130, 34_000_000
        A, B, C0 = ints(m, k), ints(k, n), ints(m, n)
        far = torch.empty((m - 1) * lda + k, dtype=torch.float64, device="cuda").as_strided((m, k), (lda, 1))
        far.copy_(A)
    else:
        N = 200 if what == "ranks" else 2700
        A, B, C0 = ints(N, N), ints(N, N), ints(N, N)

    def call(C, stream=None):
        if what == "far_rows":
            phpc.dgemm_device(far, B, C, stream=stream)
        else:
            phpc.summa_device(A, B, C, 3, 2, panel=97, mode=phpc.SUMMA_FUSED, stream=stream)

    want = C0 + (A.cpu() @ B.cpu()).cuda()  # integers: exact in any order
    C, D = C0.clone(), C0.clone()
    call(D)
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=s):
        call(C, s)
    assert torch.equal(D, want)
    X, Y, Z = ints(77, 77), ints(77, 77), ints(77, 77)
    for _ in range(3):
        C.copy_(C0)
        phpc.summa_device(X, Y, Z, 7, 7, mode=phpc.SUMMA_FUSED)  # 49 GEMMs through the buffer
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want)
