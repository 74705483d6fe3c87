"""A mixer's eval projections in one call (masters, mixes and inputs prepared and quantized, the
three GEMMs) against its ten calls, bit for bit: one batched launch of the few-row GEMM with one and
several row tiles and rounds, the other GEMM with and without K parts, four rows per wave, ragged
streams, unaligned masters, an odd count of scales a projection, and a width that keeps the ten calls."""

import pytest
import torch

from ksdraft_amd.kernels import rosa as R
from ksdraft_amd.kernels.gemm import w8a8_gemm_out
from ksdraft_amd.kernels.quant import quantize_last_dim

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,d,S,bias,offset", [
    (1, 1, 128, 1, True, 0), (2, 10, 256, 33, False, 0), (1, 301, 1536, 512, True, 0), (1, 60, 2176, 40, True, 1),
    (1, 300, 2176, 128, True, 0), (3, 701, 256, 300, False, 0), (1, 5, 1536, 2000, True, 0),
    (1, 701, 1152, 300, True, 0), (1, 5, 200, 64, True, 0)])
def test_projections_in_one_call(B, T, d, S, bias, offset, dt):
    g = torch.Generator().manual_seed(B * T + d + S)
    x = (torch.randn(B, T, d, generator=g) * 1.5).to(dt).to(DEV)
    mixes = [(torch.randn(d, generator=g) * 8).to(DEV) for _ in range(3)]  # sigmoid to its ends
    ws = [torch.randn(S * d + offset, generator=g).to(DEV)[offset:].view(S, d) for _ in range(3)]
    bs = [torch.randn(S, generator=g).to(DEV) if bias else None for _ in range(3)]
    got = R.shift_project(x, mixes, ws, bs)
    if d % 128:
        assert got is None
        return
    quant = R.shift_quantize(x, *(torch.sigmoid(m) for m in mixes))
    for y, (wq, wsc), (xq, xs), w, b in zip(*got, quant, ws, bs):
        rq, rs = quantize_last_dim(w)
        assert torch.equal(wq, rq) and torch.equal(wsc, rs)
        ref = w8a8_gemm_out(xq, xs, rq, rs, bias=b, out_dtype=dt).reshape(B, T, S)
        assert torch.equal(y, ref)
