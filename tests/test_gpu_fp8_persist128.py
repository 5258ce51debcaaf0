"""The fp8 scaled dot on 128 x 128 persistent tiles, exactly.

Integer operands (-3 .. 3) and power-of-two scales: every sum and every scaled
value is exact in fp32, so the bf16 output is its round-to-nearest-even bit for
bit.  M and N sit at tile edges (N a multiple of 8), K from two steps (fewer
than the ring's five) up; one tile, a tile per CU and, for a workgroup's
second and third tile, 564 tiles (with the fused epilogue 470: its dispatch
wants no more rounds than 256 x 128 tiles take); all format pairs.  (2049,
2056, 512) and (1023, 4104, 1152), a few tiles past a round, are left to 256 x
128 tiles.  C has padding that must stay as it was.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(65, 128, 256), (128, 136, 640), (129, 1000, 384), (700, 2040, 768),
                                   (2047, 2048, 512), (2049, 2056, 512), (1023, 4104, 1152), (1500, 6000, 512)])
@pytest.mark.parametrize("fa,fb", [(0, 0), (1, 1), (0, 1), (1, 0)])
def test_fp8_persist128_exact(tx, dev, M, N, K, fa, fb):
    dt = (torch.float8_e4m3fn, torch.float8_e5m2)
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randint(-3, 4, (M, K), generator=g).float()
    b = torch.randint(-3, 4, (N, K), generator=g).float()
    sa = torch.exp2(torch.randint(-3, 4, (M,), generator=g).float())
    sb = torch.exp2(torch.randint(-3, 4, (N,), generator=g).float())
    want = ((a @ b.t()) * sa[:, None] * sb[None, :]).to(torch.bfloat16)
    buf = torch.full((M + 1, N + 8), 7.0, dtype=torch.bfloat16, device=dev)
    out = buf[:M, :N]
    tx.dot_scaled_rowcol(a.to(dt[fa]).to(dev), sa.to(dev), b.to(dt[fb]).to(dev), sb.to(dev), out=out)
    assert torch.equal(out.cpu(), want)
    assert (buf[M] == 7.0).all() and (buf[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,N,K", [(65, 128, 256), (129, 1000, 384), (700, 2040, 768), (2049, 2056, 512),
                                   (600, 12000, 256)])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("act", [None, "relu"])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float8_e5m2])
def test_fp8_persist128_epilogue_exact(tx, dev, M, N, K, bias, act, out_dtype):
    """The same with the fused epilogue (no activation or relu: exact before
    the output's rounding), C rows of odd pitch."""
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randint(-3, 4, (M, K), generator=g).float()
    b = torch.randint(-3, 4, (N, K), generator=g).float()
    sa = torch.exp2(torch.randint(-5, -2, (M,), generator=g).float())
    sb = torch.exp2(torch.randint(-3, 1, (N,), generator=g).float())
    bv = torch.randint(-9, 10, (N,), generator=g).float() if bias else None
    y = (a @ b.t()) * sa[:, None] * sb[None, :]
    if bias:
        y = y + bv
    if act == "relu":
        y = y.clamp(min=0)
    want = (y.clamp(-57344, 57344) if out_dtype == torch.float8_e5m2 else y).to(out_dtype)
    buf = torch.zeros((M, N + 3), dtype=torch.uint8 if out_dtype == torch.float8_e5m2 else out_dtype, device=dev)
    out = buf[:, :N].view(out_dtype) if out_dtype == torch.float8_e5m2 else buf[:, :N]
    tx.dot_scaled_rowcol(a.to(torch.float8_e4m3fn).to(dev), sa.to(dev), b.to(torch.float8_e4m3fn).to(dev), sb.to(dev),
                         out=out, bias=None if bv is None else bv.to(dev), activation=act, out_dtype=out_dtype)
    assert torch.equal(out.float().cpu(), want.float())
    assert (buf[:, N:].float() == 0).all()
