"""The KS3 geometry packed from its masters in one launch against its eleven calls, bit for bit:
block remainders, both sides of softplus's threshold, zeros, large and subnormal values, infinities;
and what keeps the calls."""

import pytest
import torch
import torch.nn.functional as F

from ksdraft_amd.kernels import ks3_int8 as ki
from ksdraft_amd.kernels.quant import dequantize_last_dim, quantize_last_dim

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("Fn", [1, 255, 257, 100003])
def test_masters_packed_in_one_launch(Fn):
    g = torch.Generator().manual_seed(Fn)
    co = torch.randn(Fn, 1, 6, generator=g) * 0.05
    rs, rh = torch.randn(Fn, generator=g) * 12, torch.randn(Fn, generator=g) * 3
    edge = torch.tensor([0.0, -0.0, 20.0, 20.000002, 19.999998, 88.0, -88.0, -104.0, 1e30, -1e30, 1e-30, 1e-40,
                         float("inf"), -float("inf")])
    n = min(Fn, len(edge))
    rs[:n], rh[:n], co.view(Fn, 6)[:n, 0] = edge[:n], edge[:n], edge[:n]
    co.view(Fn, 6)[n // 2] = 0.0
    co, rs, rh = co.to(DEV), rs.to(DEV), rh.to(DEV)
    got = ki.pack_masters(co, rs, rh)
    sq, ss = ki.pack_spine(co)
    wsc, wss = quantize_last_dim((F.softplus(rs) + 1e-4).reshape(-1, 1))
    whc, whs = quantize_last_dim((0.5 * torch.tanh(rh)).reshape(-1, 1))
    want = (sq, ss, wsc, wss, whc, whs, dequantize_last_dim(wsc, wss).reshape(-1).half(),
            dequantize_last_dim(whc, whs).reshape(-1).half())
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
    assert ki.pack_masters(co.expand(Fn, 2, 6), rs, rh) is None  # rank 2
    assert ki.pack_masters(co.half(), rs, rh) is None


def test_masters_that_are_nan():
    """A NaN leaves the same codes, scale bits and fp16 values as in the eleven calls."""
    nan = float("nan")
    co = torch.full((3, 1, 6), 0.25, device=DEV)
    co[1, 0, 2] = nan
    rs, rh = torch.tensor([nan, 0.5, 30.0], device=DEV), torch.tensor([0.5, nan, -2.0], device=DEV)
    sq, ss, wsc, wss, whc, whs, sc16, sh16 = ki.pack_masters(co, rs, rh)
    want = ki.pack_spine(co)
    scale = quantize_last_dim((F.softplus(rs) + 1e-4).reshape(-1, 1))
    shift = quantize_last_dim((0.5 * torch.tanh(rh)).reshape(-1, 1))
    for a, b in ((sq, want[0]), (wsc, scale[0]), (whc, shift[0])):
        assert torch.equal(a, b)
    for a, b in ((ss, want[1]), (wss, scale[1]), (whs, shift[1])):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    for a, b in ((sc16, dequantize_last_dim(*scale)), (sh16, dequantize_last_dim(*shift))):
        assert torch.allclose(a, b.reshape(-1).half(), rtol=0, atol=0, equal_nan=True)
