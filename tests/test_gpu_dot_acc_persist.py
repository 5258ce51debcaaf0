"""D = A.B + C in fp32 on the persistent tiles (tx_dot_acc, 16-bit operands).

Operands and accumulators are small integers, so every partial sum is an
integer below 2^24 and fp32 holds it exactly: D must equal the integer result
bit for bit whatever the tile, K segment or order.  Shapes sit at the edges of
the 256-, 128- and 64-wide tiles (M one past or short of a tile, N only a
multiple of 4 or 8), with one K step short of, at and past a K segment (the
last segment one step long among them), two K steps (the fewest) and a ragged
K on the 256-wide tile.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [
    # M, N, K, layout
    (100, 260, 64 * 21, "nk"),    # 64-wide, 5 segments of 5 steps, the last one step
    (65, 264, 64 * 8, "kn"),      # 64-wide, 2 segments of 4
    (129, 4100, 64 * 9, "nk"),    # 64-wide, 2 segments, 5 + 4 steps
    (1200, 2000, 64 * 9, "nk"),   # 64-wide, 608 tiles: the segment sums start again for a second and third tile
    (1200, 2000, 64 * 9, "kn"),
    (63, 8, 128, "kn"),           # one partial tile, two K steps
    (2047, 2044, 64 * 9, "nk"),   # 128-wide, one tile per CU, 2 segments
    (2048, 2040, 64 * 9, "kn"),
    (2001, 2052, 128, "nk"),      # 128-wide, more tiles than CUs, no segments
    (4095, 4092, 192, "nk"),      # 256-wide
    (4097, 4088, 192, "kn"),      # 256-wide, a second round of tiles
    (4095, 4092, 260, "nk"),      # 256-wide, ragged K
]


@pytest.mark.parametrize("M,N,K,layout", SHAPES)
@pytest.mark.parametrize("acc", ["none", "given", "in_place"])
def test_dot_acc_persist_exact(tx, dev, M, N, K, layout, acc):
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    a = torch.randint(-3, 4, (M, K), generator=g).float()
    b = torch.randint(-3, 4, (N, K), generator=g).float()
    c = torch.randint(-1000, 1001, (M, N), generator=g).float()
    # sums below 9 K + 1000 < 2^24: exact in fp32 in any order
    want = a @ b.t() + (c if acc != "none" else 0.0)
    dt = torch.bfloat16 if K % 128 else torch.float16
    at = a.to(dt).to(dev)
    bt = (b if layout == "nk" else b.t().contiguous()).to(dt).to(dev)
    ct = None if acc == "none" else c.to(dev)
    out = torch.full((M + 1, N), 7.0, device=dev)  # one row more: nothing is written past row M - 1
    if acc == "in_place":
        out[:M] = ct
        got = tx.dot_acc(at, bt, out[:M], b_layout=layout, out=out[:M])
    else:
        got = tx.dot_acc(at, bt, ct, b_layout=layout, out=out[:M])
    assert torch.equal(got.cpu(), want)
    assert (out[M] == 7.0).all()
