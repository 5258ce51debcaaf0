"""Ragged 16-bit products on the 128- and 64-wide persistent tiles, exactly.

Integer operands (-3 .. 3): every fp32 sum is exact, so the output is its
round-to-nearest-even bit for bit.  N ends 1 .. 7 columns into an 8-column
store, rows of C have any 2-byte alignment, K is ragged (4-byte aligned rows,
read in place) or odd (padded copies), M and N sit at tile edges; the columns
and rows around C must stay as they were.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,layout", [
    (63, 65, 130, "nk"), (64, 71, 128, "nk"), (129, 1003, 66 * 2, "nk"), (500, 257, 2046, "nk"),   # 64-wide
    (1000, 801, 190, "nk"), (2001, 2047, 258, "nk"), (2048, 2041, 192, "nk"),                      # 128-wide
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
