"""Ragged 16-bit products on the 128- and 64-wide persistent tiles, exactly.

Integer operands (-3 .. 3): every fp32 sum is exact, so the output is its
round-to-nearest-even bit for bit.  N ends 1 .. 7 columns into an 8-column
store, rows of C have any 2-byte alignment, K is ragged (4-byte aligned rows,
read in place) or odd (padded copies), M and N sit at tile edges; the columns
and rows around C must stay as they were.  512 and 480 tiles on 256 CUs give a
workgroup a second tile: the ragged fetch's cursor crosses to it, and stores of
single columns come ahead of its counted waits.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,layout", [
    (63, 65, 130, "nk"), (64, 71, 128, "nk"), (129, 1003, 66 * 2, "nk"), (500, 257, 2046, "nk"),   # 64-wide
    (1000, 801, 190, "nk"), (1000, 2001, 258, "nk"),              # 64-wide, the second with 512 tiles
    (2001, 2047, 258, "nk"), (2048, 2041, 192, "nk"), (2500, 3001, 258, "nk"),  # 128-wide: 256, 256, 480 tiles
    (700, 999, 260, "kn"), (333, 777, 555, "nk"), (411, 1237, 411, "kn"),                          # copies first
    (4097, 4093, 136, "nk")])                                                                      # 256-wide
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("pad,shift", [(0, 0), (5, 1)])
def test_persist_ragged_exact(tx, dev, M, N, K, layout, dtype, pad, shift):
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randint(-3, 4, (M, K), generator=g).float()
    b = torch.randint(-3, 4, (N, K), generator=g).float()
    want = (a @ b.t()).to(dtype)
    ld = N + pad
    buf = torch.full(((M + 2) * ld + 8,), 7.0, dtype=dtype, device=dev)
    out = buf[shift + ld:shift + ld + M * ld].view(M, ld)[:, :N]
    at, bt = a.to(dtype).to(dev), b.to(dtype).to(dev)
    if layout == "nk":
        tx.dot(at, bt, out)
    else:
        tx.dot_kn(at, bt.t().contiguous(), out)
    assert torch.equal(out.cpu(), want)
    rest = buf.clone()
    rest[shift + ld:shift + ld + M * ld].view(M, ld)[:, :N] = 7.0
    assert (rest == 7.0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_odd_k_recorded_without_scratch(tx, dev, dtype):
    """An odd-K product below 1 Gi multiply-adds is recorded into a graph on a
    stream that never ran one, allocates nothing there, and later eager calls
    that do use scratch are right after the graph is gone."""
    M, N, K = 333, 777, 555
    g = torch.Generator().manual_seed(5)

    def ints(*shape):
        return torch.randint(-3, 4, shape, generator=g).float()

    a, b = torch.empty(M, K, dtype=dtype, device=dev), torch.empty(N, K, dtype=dtype, device=dev)
    out = torch.empty(M, N, dtype=dtype, device=dev)
    x, y = ints(M, K), ints(N, K)
    a.copy_(x), b.copy_(y)
    tx.dot(a, b, out)  # loads the kernels
    torch.cuda.synchronize()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    before = tx.lib.txScratchAllocations()
    with torch.cuda.graph(graph, stream=side):
        tx.dot(a, b, out)
    assert tx.lib.txScratchAllocations() == before
    for _ in range(3):
        x, y = ints(M, K), ints(N, K)
        a.copy_(x), b.copy_(y)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), (x @ y.t()).to(dtype))
    graph.reset()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        tx.dot(a, b, out)
    torch.cuda.synchronize()
    assert torch.equal(out.cpu(), (x @ y.t()).to(dtype))
