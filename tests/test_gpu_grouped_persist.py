"""The grouped fp8 dot's persistent 128 x 256 tiles (groups averaging under 192
rows), exactly.

Operands are the integers -3 .. 3 in fp8 with unit scales, so every sum is an
integer of at most 9 K (far below 2^24) and the bf16 output must be its
round-to-nearest-even bit for bit, whatever the order of K.  Group sizes sit at
the edges of a 128-row tile (empty, 1, 127, 128, 129 rows); G at and past the
512 groups that are dealt over the XCDs, 8 that are not; N ends inside a tile
and inside a column part of the last round; K from two steps (fewer than the
ring holds) up.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EDGE = [0, 1, 127, 128, 129, 0, 40]


def _sizes(groups, seed):
    g = np.random.default_rng(seed)
    s = g.choice(EDGE, size=groups)
    s[0] = 300
    return s


@pytest.mark.parametrize("groups,N,K", [(8, 264, 256), (9, 2048, 640), (16, 72, 384), (65, 520, 256), (512, 128, 256),
                                        (513, 128, 256), (40, 1032, 512)])
@pytest.mark.parametrize("fa,fb", [("e4m3fn", "e4m3fn"), ("e5m2", "e4m3fn")])
@pytest.mark.parametrize("noalloc", [False, True])
def test_grouped_persist128_exact(tx, dev, groups, N, K, fa, fb, noalloc):
    dt = {"e4m3fn": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
    sizes = _sizes(groups, groups + N + K)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    M = int(off[-1])
    assert M < 192 * groups
    g = torch.Generator().manual_seed(K + N)
    a = torch.randint(-3, 4, (M, K), generator=g).float()
    b = torch.randint(-3, 4, (groups, N, K), generator=g).float()
    aq, bq = a.to(dt[fa]).to(dev), b.to(dt[fb]).to(dev)
    sa, sb = torch.ones(M, device=dev), torch.ones(groups, N, device=dev)
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=dev)
    offd = torch.from_numpy(off).to(dev)
    if noalloc:
        from tx import _lib
        code = {"e4m3fn": _lib.FP8E4M3FN, "e5m2": _lib.FP8E5M2}
        tx.check(tx.lib.tx_dot_fp8_scaled_grouped_noalloc(
            aq.data_ptr(), code[fa], K, sa.data_ptr(), bq.data_ptr(), code[fb], K, N * K, sb.data_ptr(), N, None, 0, 0,
            out.data_ptr(), _lib.BF16, 1.0, N, offd.data_ptr(), groups, M, N, K,
            torch.cuda.current_stream().cuda_stream))
    else:
        tx.dot_scaled_rowcol_grouped(aq, sa, bq, sb, offd, out=out[:M])
    want = torch.cat([a[off[p]:off[p + 1]] @ b[p].t() for p in range(groups)]).to(torch.bfloat16)
    assert torch.equal(out[:M].cpu(), want)
    assert (out[M] == 7.0).all()
