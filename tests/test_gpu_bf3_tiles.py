"""3 x BF16 products on slice planes at the edges of their tiles, blocks and slabs: within the
FP32-accurate bound of an FP64 product, exact where every partial sum is, the same bits on every
tile shape, with everything around C untouched."""
import pytest

from conftest import phpc

pytestmark = pytest.mark.gpu


def inputs(m, k, n, seed, ints=False):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    if ints:
        return tuple(torch.randint(-8, 9, s, generator=g, device="cuda").float() for s in ((m, k), (k, n), (m, n)))
    return tuple(torch.empty(s, device="cuda").uniform_(-1, 1, generator=g) for s in ((m, k), (k, n), (m, n)))


def on_view(x, fill):
    """x as a view at an odd offset of a buffer with an odd row stride."""
    import torch
    m, n = x.shape
    buf = torch.full((m + 2, n + 5 - n % 2), fill, dtype=torch.float32, device="cuda")
    v = buf[1:1 + m, 1:1 + n]
    v.copy_(x)
    return buf, v


def check(A, B, C0, C):
    k = A.shape[1]
    want = C0.double() + A.double() @ B.double()
    mag = C0.double().abs() + A.double().abs() @ B.double().abs()
    assert bool(((C.double() - want).abs() <= ((k + 2) * 2.0 ** -24 + 2.0 ** -23) * mag).all()), (A.shape, B.shape)


def run_plan(cfg, items):
    import torch
    phpc.set_tuning(8, cfg)
    try:
        plan = phpc.Plan(phpc.F32X3, items)
    finally:
        phpc.set_tuning(8, -1)
    assert plan.info()["config"] == cfg
    plan.launch()
    torch.cuda.synchronize()
    plan.close()


# one off the tiles' edges and the blocks' (32 rows, 16 k); k below, at and past the ring's three
# slabs and past the steady loop's first turn (nine)
EDGES = [(1, 1, 1), (31, 15, 33), (33, 16, 31), (63, 17, 65), (65, 32, 64), (127, 47, 129), (129, 48, 255),
         (257, 49, 127), (128, 143, 128), (64, 144, 64), (100, 161, 300), (40, 400, 31)]


@pytest.mark.parametrize("cfg", [4, 5, 6])
def test_plan_edges(cfg):
    import torch
    for ints in (False, True):
        ops, items, bufs = [], [], []
        for i, (m, k, n) in enumerate(EDGES):
            A, B, C0 = inputs(m, k, n, 100 + i, ints)
            # what surrounds the operands is NaN: an entry of padding that reached an output would show
            bA, bB, bC = on_view(A, float("nan")), on_view(B, float("nan")), on_view(C0, 7.0)
            ops.append((A, B, C0))
            bufs.append((bA[0], bB[0], bC[0]))
            items.append((bA[1], bB[1], bC[1]))
        run_plan(cfg, items)
        for (A, B, C0), (_, _, C), (_, _, buf) in zip(ops, items, bufs):
            if ints:
                assert torch.equal(C, C0 + A @ B)
            check(A, B, C0, C)
            C.fill_(7.0)
            assert torch.all(buf == 7.0)


# one product through each tile rule (64x64; 128x64 with a 64x64 tail; 128x128 with one by rows
# and by columns; 256x128), against every pinned plan's bits
@pytest.mark.parametrize("m,k,n", [(1025, 130, 1023), (1500, 150, 1477), (2801, 140, 2601), (2601, 129, 2801),
                                   (4096, 300, 2048)])
def test_single_product_equals_plans(m, k, n):
    import torch
    A, B, C0 = inputs(m, k, n, m + n)
    C = C0.clone()
    phpc.sgemm_device(A, B, C, method=phpc.SGEMM_BF16X3)
    torch.cuda.synchronize()
    check(A, B, C0, C)
    for cfg in (4, 5, 6):
        D = C0.clone()
        run_plan(cfg, [(A, B, D)])
        assert torch.equal(C.view(torch.int32), D.view(torch.int32)), cfg


# the in-register kernel: 64x64 tiles below one 128x128 tile per CU
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (63, 31, 65), (65, 33, 127), (129, 64, 64), (500, 100, 300),
                                   (2100, 60, 2300)])
def test_in_register_tiles(m, k, n):
    import torch
    A, B, C0 = inputs(m, k, n, 3)
    _, dA = on_view(A, float("nan"))
    _, dB = on_view(B, float("nan"))
    buf, dC = on_view(C0, 7.0)
    phpc.sgemm_device(dA, dB, dC, method=phpc.SGEMM_BF16X3)
    torch.cuda.synchronize()
    check(A, B, C0, dC)
    D = C0.clone()
    run_plan(2, [(A, B, D)])
    assert torch.equal(dC, D)
    dC.fill_(7.0)
    assert torch.all(buf == 7.0)


def test_captured_product_takes_no_workspace():
    """A product that takes the shared planes in eager calls is captured as the in-register
    kernel, and replays between eager calls on other sizes give the same result."""
    import torch
    A, B, C0 = inputs(1100, 300, 1000, 9)
    C = C0.clone()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        phpc.sgemm_device(A, B, C, method=phpc.SGEMM_BF16X3)
    first = None
    for rep in range(3):
        C.copy_(C0)
        X, Y, Z = inputs(1300 + 300 * rep, 400, 1200, rep)
        phpc.sgemm_device(X, Y, Z, method=phpc.SGEMM_BF16X3)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        check(A, B, C0, C)
        first = C.clone() if first is None else first
        assert torch.equal(C, first)


def test_smaller_products_leave_a_captured_large_one_alone():
    """A captured large product keeps its planes: eager products below its size, with planes larger
    than all before, run between its replays."""
    import torch
    A, B, C0 = inputs(2048, 256, 2048, 1)
    C, want = C0.clone(), C0.clone()
    phpc.sgemm_device(A, B, want, method=phpc.SGEMM_BF16X3)  # allocates the planes
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        phpc.sgemm_device(A, B, C, method=phpc.SGEMM_BF16X3)
    held = []
    for rep in range(3):
        C.copy_(C0)
        X, Y, Z = inputs(1500, 2000 * (rep + 1), 1500, rep)
        Z0 = Z.clone()
        phpc.sgemm_device(X, Y, Z, method=phpc.SGEMM_BF16X3)
        held.append(torch.full((4 << 20,), float("nan"), device="cuda"))  # would take freed planes' place
        torch.cuda.synchronize()
        check(X, Y, Z0, Z)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want)


def test_products_on_several_streams():
    """More streams than workspaces, two rounds, planes of several sizes, one stream's beyond the
    size that goes to the first workspace."""
    import torch
    shapes = [(1500, 300, 1500), (1100, 700, 1000), (1024, 1024, 1024), (1300, 140, 1700), (1025, 2000, 1030),
              (1500, 64000, 1500)]
    ops = [inputs(*sh, seed=i) for i, sh in enumerate(shapes)]
    alone = []
    for A, B, C0 in ops:
        C = C0.clone()
        phpc.sgemm_device(A, B, C, method=phpc.SGEMM_BF16X3)
        torch.cuda.synchronize()
        alone.append(C)
    streams = [torch.cuda.Stream() for _ in ops]
    outs = [[C0.clone() for _, _, C0 in ops] for _ in range(2)]
    torch.cuda.synchronize()
    for out in outs:
        for s, (A, B, _), C in zip(streams, ops, out):
            phpc.sgemm_device(A, B, C, method=phpc.SGEMM_BF16X3, stream=s)
    torch.cuda.synchronize()
    for out in outs:
        for C, want in zip(out, alone):
            assert torch.equal(C, want)


# one call, one result: the in-register kernel (64x64 and 128x128 tiles, 16-byte and 4-byte loads)
# sums as the planes' does
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (31, 15, 33), (65, 33, 127), (128, 200, 64), (300, 1000, 500),
                                   (1025, 130, 1023), (2048, 96, 2048), (2101, 161, 2303)])
def test_in_register_bits_are_the_planes(m, k, n):
    import torch
    A, B, C0 = inputs(m, k, n, 5 * m + n)
    out = []
    for cfg in (2, 4):
        C = C0.clone()
        run_plan(cfg, [(A, B, C)])
        out.append(C.view(torch.int32))
    assert torch.equal(*out)


@pytest.mark.parametrize("m,k,n", [(1100, 300, 1000), (2000, 257, 2001)])
def test_captured_bits_are_the_eager(m, k, n):
    import torch
    A, B, C0 = inputs(m, k, n, m)
    want, C = C0.clone(), C0.clone()
    phpc.sgemm_device(A, B, want, method=phpc.SGEMM_BF16X3)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        phpc.sgemm_device(A, B, C, method=phpc.SGEMM_BF16X3)
    for _ in range(3):
        C.copy_(C0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(C.view(torch.int32), want.view(torch.int32))


# either side of the rule between planes and the in-register kernel, with 128x128 tiles in whole
# rounds and the rest apart (by columns, by rows)
@pytest.mark.parametrize("m,k,n", [(100, 70, 40000), (20000, 65, 200), (256, 1024, 8192), (256, 2100, 8192),
                                   (257, 511, 4100), (257, 512, 4100), (2047, 130, 2047)])
def test_products_beside_the_rule(m, k, n):
    import torch
    A, B, C0 = inputs(m, k, n, m + k)
    C, D = C0.clone(), C0.clone()
    phpc.sgemm_device(A, B, C, method=phpc.SGEMM_BF16X3)
    torch.cuda.synchronize()
    check(A, B, C0, C)
    run_plan(4, [(A, B, D)])
    assert torch.equal(C.view(torch.int32), D.view(torch.int32))


@pytest.mark.parametrize("shapes", [[(100, 40, 40000)], [(90, 33, 300), (2000, 64, 2100), (200, 50, 5000)],
                                    [(i % 90 + 1, 20 + i, 70) for i in range(300)]])
def test_in_register_plan_in_two_launches(shapes):
    import torch
    ops = [inputs(*s, seed=i) for i, s in enumerate(shapes)]
    outs = []
    for cfg in (2, 4):
        items = [(A, B, C.clone()) for A, B, C in ops]
        run_plan(cfg, items)
        outs.append([C for _, _, C in items])
    for (A, B, C0), C, D in zip(ops, *outs):
        check(A, B, C0, C)
        assert torch.equal(C.view(torch.int32), D.view(torch.int32))
