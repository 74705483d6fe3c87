"""The persistent group-128 GEMM on ragged shapes that lie past the few-row kernel's rule: both
epilogues (K in one part and in several), every output type, bias, residual (also in place), the
saturating store and subnormal scales, bit for bit against the oracle's ordered contract."""

import ctypes

import numpy as np
import pytest
import torch

from ksdraft_amd import _lib
from ksdraft_amd.kernels import gemm as kg
from oracle import gemm as og
from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("mag", [1.0, 1e-4])
@pytest.mark.parametrize("M,N,K,splits", [(300, 1043, 256, 1), (257, 1291, 640, 1), (4097, 33, 384, 1),
                                          (300, 1043, 2048, 2), (641, 515, 2304, 2), (65, 129, 8192, 8)])
def test_persistent_gemm(M, N, K, splits, mag):
    few = ctypes.c_int(-1)
    _lib.call("ksd_w8a8_gemm_few_rows", M, N, K, ctypes.byref(few))
    assert few.value == 0 and kg.gemm_splits(M, N, K) == splits == og.splits_for(M, N, K)
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K, generator=g) * mag, torch.randn(N, K, generator=g) * 0.1
    a[::5] *= 3e5  # past the fp16 range
    ops = (*oq.quantize_last_dim(a.numpy()), *oq.quantize_last_dim(w.numpy()))
    dev = [torch.from_numpy(np.ascontiguousarray(o)).to(DEV) for o in ops]
    bias = torch.randn(N, generator=g)
    ref = torch.from_numpy(og.gemm_ordered(*ops))
    refb = torch.from_numpy(og.gemm_ordered(*ops, bias=bias.numpy()))
    assert torch.equal(kg.w8a8_gemm(*dev).cpu(), ref)
    for dt in (torch.float32, torch.bfloat16, torch.float16):
        y = kg.w8a8_gemm_out(*dev, bias=bias.to(DEV), out_dtype=dt)
        assert torch.equal(y.cpu(), refb.to(dt)), dt
        r = torch.randn(M, N, generator=g).to(dt)
        rd = r.to(DEV)
        assert torch.equal(kg.w8a8_gemm_out(*dev, bias=bias.to(DEV), out_dtype=dt, residual=rd).cpu(), r + refb.to(dt)), dt
        kg.w8a8_gemm_out(*dev, bias=bias.to(DEV), out_dtype=dt, residual=rd, out=rd)
        assert torch.equal(rd.cpu(), r + refb.to(dt)), dt
    assert torch.equal(kg.w8a8_gemm_out(*dev, fp16_saturate=True).cpu(), ref.half().clamp(-65504, 65504))
