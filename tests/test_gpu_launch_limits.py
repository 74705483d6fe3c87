"""Calls past the 2^32 threads that one launch holds: K padding of 64 GiB of codes, and an int8
linear whose two quantizations fit a launch each but not one together."""

import pytest
import torch

from ksdraft_amd import _lib
from ksdraft_amd.kernels import Int8Linear
from ksdraft_amd.kernels.gemm import _pad_operands, w8a8_gemm_out
from ksdraft_amd.kernels.quant import quantize_last_dim

pytestmark = pytest.mark.gpu
DEV = "cuda"
GiB = 1 << 30


@pytest.fixture(autouse=True)
def _give_back():
    yield
    torch.cuda.empty_cache()


def _need(gib):
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < gib * GiB:
        pytest.skip(f"needs {gib} GiB of free device memory")


@pytest.mark.parametrize("rows", [5, (1 << 29) + 3])
def test_pad_codes(rows):
    if rows > 5:
        _need(72)
    a = torch.arange(rows, device=DEV).to(torch.int8).view(rows, 1)
    b = torch.arange(70, device=DEV, dtype=torch.int8).view(2, 35)
    pa, pb = _pad_operands(_lib.require_gpu(a), (a, b), (128, 128))
    assert torch.equal(pb, torch.nn.functional.pad(b, (0, 93)))
    for r in range(0, rows, 1 << 25):
        part = pa[r:r + (1 << 25)]
        assert torch.equal(part[:, :1], a[r:r + (1 << 25)])
        assert not bool(part[:, 1:8].any()) and not bool(part.view(torch.int64)[:, 1:].any())


@pytest.mark.parametrize("M", [48, (1 << 28) - 16])
def test_int8_linear_rows(M):
    if M > 48:
        _need(110)
    g = torch.Generator(device=DEV).manual_seed(1)
    lin = Int8Linear(128, 1, bias=False).to(DEV).eval()
    head = torch.randn(16, 128, generator=g, device=DEV).bfloat16()
    x = torch.zeros(M, 128, dtype=torch.bfloat16, device=DEV)
    x[:16], x[-16:] = head, head.flip(0)
    with torch.no_grad():
        lin.weight.copy_(torch.randn(1, 128, generator=g, device=DEV))
        y = lin(x)
        want = w8a8_gemm_out(*quantize_last_dim(head), *quantize_last_dim(lin.weight), out_dtype=torch.bfloat16)
    assert torch.equal(y[:16], want) and torch.equal(y[-16:], want.flip(0)) and not bool(y[16:-16].any())
