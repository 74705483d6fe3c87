"""The KS3 spines without a table, and the table readers' row split, against the oracle, bit for bit."""

import numpy as np
import pytest
import torch

from ksdraft_amd.kernels import ks3_int8 as ki
from oracle import ks3 as ok
from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _spine(M, Fn, seed):
    r = np.random.default_rng(seed)
    x = (r.standard_normal((M, Fn)) * 6).astype(np.float32)
    x[r.random((M, Fn)) < 0.02] *= 1e5  # past the LUT's domain and the fp16 range
    lut = ki.make_tanh_lut("cpu").numpy()
    return x, (r.integers(-127, 128, (Fn, 6)).astype(np.int8), (r.random(Fn) * 0.01).astype(np.float16),
               (r.random(Fn) + 0.2).astype(np.float16), (r.standard_normal(Fn) * 0.3).astype(np.float16), lut)


# one row, ragged segments and row blocks, odd widths; (3700, 1984) and (3703, 1985) lie past the
# table-free rule: the table readers, their row split no longer 512; the last four lie on either
# side of it (fused and ragged rows 600 + 3.4e6 / 128-chart columns, composed 460 + 1.2e6)
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("M,Fn", [(1, 1), (7, 130), (9, 128), (33, 257), (3700, 1984), (3703, 1985),
                                  (13881, 130), (13882, 130), (5147, 256), (5148, 256)])
def test_spines_without_a_table(M, Fn, group):
    x, par = _spine(M, Fn, M + Fn)
    dev = [_t(p) for p in par]
    rows = np.unique(np.r_[0:min(M, 40), max(0, M - 40):M, np.arange(0, M, 97)])
    q, s = ki.spine_fused_int8(_t(x), *dev, group)
    oq_, os_ = ok.spine_fused_int8(x[rows], *par, group)
    assert np.array_equal(q[rows].cpu().numpy(), oq_) and np.array_equal(s[rows].cpu().numpy(), os_)
    c16 = np.clip(x, -65504, 65504).astype(np.float16)
    h, q, s = ki.spine_int8(_t(c16), *dev, group, want_h=True)
    oh = np.asarray(ok.spine_features_int8(c16[rows], *par), np.float32)
    oq_, os_ = oq.quantize_last_dim(oh, group)
    assert np.array_equal(h[rows].cpu().numpy(), oh)
    assert np.array_equal(q[rows].cpu().numpy(), oq_) and np.array_equal(s[rows].cpu().numpy(), os_)
