"""The int8 linear in one call (master and tokens quantized in one launch, then the GEMM) against
its three calls, bit for bit: aligned, strided and unaligned tokens, K parts, a K that keeps the three
calls, and one and four rows per wave on either side."""

import pytest
import torch

from ksdraft_amd.kernels import Int8Linear
from ksdraft_amd.kernels.gemm import w8a8_gemm_out
from ksdraft_amd.kernels.quant import quantize_last_dim

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N,bias,res", [(1, 128, 1, True, False), (17, 1536, 100, False, True), (300, 2176, 520, True, True),
                                            (5000, 256, 40, True, False), (3, 200, 64, True, True)])
def test_int8_linear_in_one_call(M, K, N, bias, res, dt):
    g = torch.Generator().manual_seed(M + K)
    lin = Int8Linear(K, N, bias=bias).to(DEV).eval()
    with torch.no_grad():
        lin.weight.copy_(torch.randn(N, K, generator=g))
        if bias:
            lin.bias.copy_(torch.randn(N, generator=g))
    wide = torch.randn(M, K + 3, generator=g).to(dt).to(DEV)
    r = torch.randn(M, N, generator=g).to(dt).to(DEV) if res else None
    wq, ws = quantize_last_dim(lin.weight.detach())
    for x in (wide[:, :K].contiguous(), wide[:, :K], wide[:, 1:K + 1]):  # aligned, strided, unaligned
        ref = w8a8_gemm_out(*quantize_last_dim(x), wq, ws, bias=None if lin.bias is None else lin.bias.detach(),
                            out_dtype=dt, residual=r)
        with torch.no_grad():
            y = lin(x, r)
        assert torch.equal(y, ref)
        assert torch.equal(lin.weight_codes, wq) and torch.equal(lin.weight_scales, ws)


# four rows a wave from 1024 blocks of 16 rows and 512 columns: x alone, the master alone, both
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(16385, 128, 24), (5, 128, 16390), (16387, 128, 16386), (17, 1536, 100)])
def test_rows_per_wave_and_strided_rows(M, K, N, dt):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    lin = Int8Linear(K, N, bias=False).to(DEV).eval()
    wide = torch.randn(M, K + 8, generator=g, device=DEV).to(dt)
    with torch.no_grad():
        lin.weight.copy_(torch.randn(N, K, generator=g, device=DEV))
    wq, ws = quantize_last_dim(lin.weight.detach())
    for x in (wide[:, :K].contiguous(), wide[:, :K], wide[:, 8:]):  # dense, and 16-byte aligned rows 8 apart
        ref = w8a8_gemm_out(*quantize_last_dim(x.contiguous()), wq, ws, out_dtype=dt)
        with torch.no_grad():
            y = lin(x)
        assert torch.equal(y, ref)
        assert torch.equal(lin.weight_codes, wq) and torch.equal(lin.weight_scales, ws)
