"""The few-row GEMM kernel against the oracle's ordered contract, bit for bit: row and column
remainders of its 16-wide tiles, every row-tile count, several rounds of groups, K parts, each
output type with bias and residual, and both sides of the rule that selects it."""

import numpy as np
import pytest
import torch

from ksdraft_amd.kernels import gemm as kg
from oracle import gemm as og
from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _np(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16) if t.element_size() == 2 else t.cpu().numpy().view(np.uint32)


# (16, 520, 2176): 17 groups in two rounds, 2 K parts; (7, 40, 5888): 46 groups, 5 K parts;
# (65, 1040, 128), (256, 256, 256): MT = 4 with several row blocks; the last two lie past the rule
@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (16, 16, 128), (17, 15, 640), (33, 31, 1536), (64, 100, 2048),
                                   (16, 520, 2176), (7, 40, 5888), (65, 1040, 128), (256, 256, 256), (1, 4100, 512),
                                   (33, 40, 2176), (300, 1040, 256)])
def test_few_rows_bit_exact(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g) * 0.1
    ops = (*oq.quantize_last_dim(a.numpy()), *oq.quantize_last_dim(w.numpy()))
    dev = [torch.from_numpy(np.ascontiguousarray(o)).to(DEV) for o in ops]
    bias = torch.randn(N, generator=g)
    ref = og.gemm_ordered(*ops)
    assert np.array_equal(_np(kg.w8a8_gemm(*dev)), ref.view(np.uint32))
    refb = torch.from_numpy(og.gemm_ordered(*ops, bias=bias.numpy()))
    for dt in (torch.float32, torch.bfloat16, torch.float16):
        res = torch.randn(M, N, generator=g).to(dt)
        y = kg.w8a8_gemm_out(*dev, bias=bias.to(DEV), out_dtype=dt)
        assert np.array_equal(_np(y), _np(refb.to(dt)))
        y = kg.w8a8_gemm_out(*dev, bias=bias.to(DEV), out_dtype=dt, residual=res.to(DEV))
        assert np.array_equal(_np(y), _np(res + refb.to(dt)))
    y = kg.w8a8_gemm_out(*dev, fp16_saturate=True)
    assert np.array_equal(_np(y), _np(torch.from_numpy(ref).half().clamp(-65504, 65504)))
