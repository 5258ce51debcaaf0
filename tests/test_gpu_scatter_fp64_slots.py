"""fp32 scatter-add through fp64 LDS slots, exactly.

Values are the integers -3 .. 3, so every bin's sum is an integer below 2^24
and any order of additions gives it exactly: bins must equal the integer
result bit for bit.  Bin counts sit at the edges of what one fp64 table holds
(18,432), of a mixed fp64 / fp32 window (34,816) and past one window; keys are
Zipf (the hot block first or moved to the middle of the range) or flat, with
out-of-range keys, a mask, misaligned buffers and a length that is no multiple
of a workgroup's step.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(tx, dev, n, nbins, zipf, seed, shift=0, mask=False, offset=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    if zipf:
        cdf = np.cumsum(np.arange(1, nbins + 1, dtype=np.float64) ** -1.1)
        cdf = torch.from_numpy(cdf / cdf[-1]).to(dev)
        u = torch.rand(n + offset, generator=g, device=dev, dtype=torch.float64)
        idx = (torch.searchsorted(cdf, u, right=True).clamp_(max=nbins - 1) + shift) % nbins
    else:
        idx = torch.randint(0, nbins, (n + offset,), generator=g, device=dev)
    idx = idx.to(torch.int32)
    idx[offset + 5::1000] = -1          # dropped
    idx[offset + 7::1000] = nbins       # dropped
    val = torch.randint(-3, 4, (n + offset,), generator=g, device=dev).float()
    idx, val = idx[offset:], val[offset:]
    m = (torch.rand(n, generator=g, device=dev) < 0.9).to(torch.uint8) if mask else None
    bins = torch.randint(-9, 10, (nbins,), generator=g, device=dev).float()
    keep = (idx >= 0) & (idx < nbins) & (True if m is None else m != 0)
    ki, kv = idx[keep].cpu().numpy(), val[keep].cpu().numpy()
    want = bins.cpu().numpy().astype(np.float64) + np.bincount(ki, weights=kv, minlength=nbins)
    assert np.abs(want).max() < 1 << 24
    tx.atomic_rmw("fadd", bins, idx, val, mask=m)
    assert np.array_equal(bins.cpu().numpy().astype(np.float64), want)


@pytest.mark.parametrize("nbins", [1, 63, 2048, 18431, 18432, 18433])
@pytest.mark.parametrize("n,mask,offset", [(1, False, 0), (12289, True, 0), (1_000_003, False, 1), (3_200_000, True, 0)])
def test_fp64_table(tx, dev, nbins, n, mask, offset):
    _run(tx, dev, n, nbins, n % 2 == 0, nbins + n, mask=mask, offset=offset)


@pytest.mark.parametrize("nbins", [18433, 20480, 34815, 34816, 34817])
@pytest.mark.parametrize("zipf,shift", [(True, 0), (True, 15000), (False, 0)])
def test_mixed_table_one_window(tx, dev, nbins, zipf, shift):
    # 128 Ki updates per workgroup: the mixed table is considered (flat keys refuse it)
    _run(tx, dev, 131072 * 256 + 4099, nbins, zipf, nbins + shift, shift=shift)


@pytest.mark.parametrize("nbins", [36865, 65536, 147456])
@pytest.mark.parametrize("shift,mask", [(0, False), (30001, True), (34000, False)])
def test_mixed_window_with_spill(tx, dev, nbins, shift, mask):
    _run(tx, dev, 49152 * 256 + 77, nbins, True, nbins + shift, shift=shift, mask=mask)
