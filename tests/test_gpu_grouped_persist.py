"""The grouped fp8 dot's persistent 128 x 256 tiles (groups averaging under 192
rows), exactly.

Operands are the integers -3 .. 3 in fp8 with unit scales, so every sum is an
integer of at most 9 K (far below 2^24) and the bf16 output must be its
round-to-nearest-even bit for bit, whatever the order of K.  Group sizes sit at
the edges of a 128-row tile (empty, 1, 127, 128, 129 rows); from 8 to 513
groups, and with 512 MiB of weights 9 to 129, which are dealt over the XCDs up
to 128; N ends inside a tile
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


def test_grouped_without_a_map(tx, dev):
    """4096 groups of 0 .. 2 rows through the no-allocation entry point: the m
    tiles' map does not fit its 64 KiB workspace, so the tiles (whose K starts
    at the expert's own step, in column parts) search the prefix."""
    groups, N, K = 4096, 8, 256
    g = np.random.default_rng(3)
    off = np.concatenate([[0], np.cumsum(g.integers(0, 3, groups))]).astype(np.int32)
    M = int(off[-1])
    assert groups + 1 + 4 * (M // 128 + groups) > 16384
    gen = torch.Generator().manual_seed(9)
    a = torch.randint(-3, 4, (M, K), generator=gen).float()
    b = torch.randint(-3, 4, (groups, N, K), generator=gen).float()
    want = torch.bmm(a[:, None], b[np.repeat(np.arange(groups), np.diff(off))].transpose(1, 2).contiguous())
    aq, bq = a.to(torch.float8_e4m3fn).to(dev), b.to(torch.float8_e4m3fn).to(dev)
    sa, sb = torch.ones(M, device=dev), torch.ones(groups, N, device=dev)
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=dev)
    offd = torch.from_numpy(off).to(dev)
    from tx import _lib
    tx.check(tx.lib.tx_dot_fp8_scaled_grouped_noalloc(
        aq.data_ptr(), _lib.FP8E4M3FN, K, sa.data_ptr(), bq.data_ptr(), _lib.FP8E4M3FN, K, N * K, sb.data_ptr(), N,
        None, 0, 0, out.data_ptr(), _lib.BF16, 1.0, N, offd.data_ptr(), groups, M, N, K,
        torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out[:M].cpu(), want[:, 0].to(torch.bfloat16))
    assert (out[M] == 7.0).all()


@pytest.mark.parametrize("groups", [7, 16])
def test_grouped_overlapping_groups(tx, dev, groups):
    """Offsets that go back to 0 give every second group all the rows: more m
    tiles than the map has room for, so the scan is done again without dealing
    and the tiles search the prefix.  All groups share one expert's weights,
    so every group that writes a row writes the same values."""
    M, N, K = 1000, 520, 384
    off = np.array([0 if p % 2 == 0 else M for p in range(groups + 1)], np.int32)
    m_tiles, room = (groups + 1) // 2 * 8, 8 + groups
    assert M < 192 * groups and m_tiles > room
    gen = torch.Generator().manual_seed(11)
    a = torch.randint(-3, 4, (M, K), generator=gen).float()
    b = torch.randint(-3, 4, (N, K), generator=gen).float()
    aq = a.to(torch.float8_e4m3fn).to(dev)
    bq = b.to(torch.float8_e4m3fn).to(dev).expand(groups, N, K).contiguous()
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=dev)
    tx.dot_scaled_rowcol_grouped(aq, torch.ones(M, device=dev), bq, torch.ones(groups, N, device=dev),
                                 torch.from_numpy(off).to(dev), out=out[:M])
    assert torch.equal(out[:M].cpu(), (a @ b.t()).to(torch.bfloat16))
    assert (out[M] == 7.0).all()


@pytest.mark.parametrize("groups,N,K", [(9, 16384, 4096), (16, 8192, 4096), (65, 2064, 4096), (128, 1032, 4096),
                                        (129, 1024, 4096)])
def test_grouped_dealt(tx, dev, groups, N, K):
    """Weights of 512 MiB and more: the map holds the groups dealt over the
    XCDs by falling tile count (not past 128 groups).  Skewed sizes with empty
    groups, from 40 to 800 rows for the largest; the reference in fp32 on the
    GPU, a group at a time (integers: exact)."""
    assert groups * N * K >= 1 << 29
    g = np.random.default_rng(groups)
    sizes = g.permutation((900 / np.arange(2, groups + 2) ** 1.1).astype(np.int64))
    sizes[[1, 3]] = 0
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    M = int(off[-1])
    assert M < 192 * groups
    gen = torch.Generator(device=dev).manual_seed(groups)
    a = torch.randint(-3, 4, (M, K), generator=gen, device=dev, dtype=torch.int8).float().to(torch.float8_e4m3fn)
    b = torch.empty((groups, N, K), dtype=torch.float8_e4m3fn, device=dev)
    for p in range(groups):
        b[p] = torch.randint(-3, 4, (N, K), generator=gen, device=dev, dtype=torch.int8).float().to(torch.float8_e4m3fn)
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=dev)
    tx.dot_scaled_rowcol_grouped(a, torch.ones(M, device=dev), b, torch.ones(groups, N, device=dev),
                                 torch.from_numpy(off).to(dev), out=out[:M])
    for p in range(groups):
        if sizes[p]:
            want = (a[off[p]:off[p + 1]].float() @ b[p].float().t()).to(torch.bfloat16)
            assert torch.equal(out[off[p]:off[p + 1]], want), p
    assert (out[M] == 7.0).all()
