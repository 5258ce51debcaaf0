"""The row-wise quantiser's 1024-thread rows: codes and scales bit for bit
against the oracle, at the row lengths and counts where the kernel changes
(quant_row_wide: K from 2048 fp32 / 6144 bf16 with at most a row per CU, longer
with more rows, up to 16384), with vectors left over for some threads only, and
the lengths that stay on the other paths."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,K", [(1, 2056), (3, 4096), (511, 2304), (512, 2304), (5, 2048), (700, 8192),
                                    (700, 8200), (5, 16384), (2, 16392), (2, 8191), (600, 1028), (4, 16380),
                                    (256, 6144), (257, 6152), (256, 6136), (300, 8200), (600, 13320), (600, 10240),
                                    (2048, 11272), (1024, 8196)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("fmt", [1, 2])
def test_rowwise_wide_exact(tx, oracle, dev, rows, K, dtype, fmt):
    g = torch.Generator().manual_seed(rows * 31 + K)
    x = (torch.randn(rows, K, generator=g) * torch.exp2(torch.randint(-8, 9, (rows, 1), generator=g).float())).to(dtype)
    x[0, K - 1] = 1000.0  # the row's largest in its last element
    q, s = tx.quantize_rowwise(x.to(dev), {1: torch.float8_e4m3fn, 2: torch.float8_e5m2}[fmt])
    xh = x.numpy() if dtype == torch.float32 else x.view(torch.int16).numpy().view(np.uint16)
    rq, rs = oracle.quant_rowwise(xh, fmt)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), rq)
    assert np.array_equal(s.cpu().numpy().view(np.uint32), rs.view(np.uint32))
