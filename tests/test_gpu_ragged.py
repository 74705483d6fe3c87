"""Rows of any length and alignment: the dual quantizers' ragged form (one pass where C % 8 != 0
or the rows are not 16-byte aligned) and the one-launch zero padding of GEMM operands, bit-exact
against the oracle."""

import numpy as np
import pytest
import torch

from ksdraft_amd.kernels.gemm import w8a8_gemm, w8a8_gemm_pair
from ksdraft_amd.kernels.quant import (quantize_dual, quantize_dual2, quantize_dual_colsum,
                                       quantize_last_dim)
from ksdraft_amd.train import cross_entropy_int8
from oracle import gemm as og
from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DT = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def _ragged(R, C, dt, seed, offset=0):
    """(R, C) whose base lies `offset` elements past an allocation's start."""
    g = torch.Generator().manual_seed(seed)
    buf = torch.randn(R * C + offset, generator=g).to(DT[dt]).to(DEV)
    return buf[offset:].view(R, C)


def _eq(got, want):
    for a, b in zip(got, want):
        assert np.array_equal(a.cpu().numpy().view(np.uint8), np.ascontiguousarray(b).view(np.uint8))


@pytest.mark.parametrize("dt", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("R,C,offset", [(1, 1, 0), (3, 7, 0), (128, 129, 0), (131, 127, 1), (257, 135, 3),
                                        (64, 136, 1), (5, 777, 0)])
def test_dual_quantizers_of_ragged_rows(R, C, offset, dt):
    x = _ragged(R, C, dt, 5, offset)
    xf = x.float().cpu().numpy()
    row, col = oq.quantize_last_dim(xf), oq.quantize_transpose(xf)
    _eq(quantize_dual(x), (*row, *col))
    xt = oq.requant_transpose(*row)
    _eq(quantize_dual(x, t_from_codes=True), (*row, *xt))
    w = _ragged(2, C, dt, 6)
    wrow = oq.quantize_last_dim(w.float().cpu().numpy())
    a, b = quantize_dual2(w, x)
    _eq(a, (*wrow, *oq.requant_transpose(*wrow)))
    _eq(b, (*row, *xt))
    *q, s = quantize_dual_colsum(x)
    _eq(q, (*row, *col))
    # R fp32 adds in any order: below R * 2^-23 of the sum of magnitudes
    ref = xf.astype(np.float64).sum(0)
    assert (np.abs(s.cpu().numpy() - ref) <= R * 2.0 ** -23 * np.abs(xf).sum(0) + 1e-30).all()


@pytest.mark.parametrize("R,V", [(1, 3), (130, 257), (5, 1001)])
def test_cross_entropy_gradient_of_ragged_vocabularies(R, V):
    g = torch.Generator().manual_seed(7)
    y = torch.randn(R, V, generator=g).to(DEV)
    t = torch.randint(0, V, (R,), generator=g).to(DEV)
    loss, ops, dy = cross_entropy_int8(y, t, grad_output=64.0, return_dy=True)
    y64 = y.double().requires_grad_(True)
    ref = torch.nn.functional.cross_entropy(y64, t)
    gref, = torch.autograd.grad(ref, y64, torch.tensor(64.0, dtype=torch.float64, device=DEV))
    assert abs(float(loss) - float(ref.detach())) <= 2e-5 * abs(float(ref.detach()))
    assert float((dy.double() - gref).abs().max()) <= 1e-5 * 64.0 / R
    d = dy.cpu().numpy()
    _eq(ops, (*oq.quantize_last_dim(d), *oq.quantize_transpose(d)))
    _eq(cross_entropy_int8(y, t, grad_output=64.0)[1], [o.cpu().numpy() for o in ops])


@pytest.mark.parametrize("K0,K1", [(1, 128), (16, 127), (129, 1000), (640, 33)])
def test_gemm_operands_padded_in_one_launch(K0, K1):
    g = torch.Generator().manual_seed(8)
    probs, want = [], []
    for M, N, K in ((5, 130, K0), (129, 7, K1)):
        a, w = (torch.randn(r, K, generator=g) for r in (M, N))
        qa, qw = quantize_last_dim(a.to(DEV)), quantize_last_dim(w.to(DEV))
        ref = og.gemm_ordered(*oq.quantize_last_dim(a.numpy()), *oq.quantize_last_dim(w.numpy()))
        assert np.array_equal(w8a8_gemm(*qa, *qw).cpu().numpy(), ref)
        probs.append((*qa, *qw, torch.float32))
        want.append(ref)
    for y, ref in zip(w8a8_gemm_pair(*probs), want):
        assert np.array_equal(y.cpu().numpy(), ref)
