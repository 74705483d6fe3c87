"""An eval mixer with more streams than the one-launch products take keeps the torch ops."""

import pytest
import torch

from ksdraft_amd.kernels import Int8Linear
from ksdraft_amd.kernels import rosa as R
from ksdraft_amd.model.rosa import RosaMixer

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("S", [64 * 65535, 64 * 65535 + 1])
def test_eval_mixer_past_the_products_grid(S):
    g = torch.Generator(device=DEV).manual_seed(3)
    with torch.device(DEV):
        mix = RosaMixer(8, S).eval()
        x = torch.randn(1, 3, 8, generator=g)
    with torch.no_grad():
        mix.payload.copy_(1 + 0.1 * torch.randn(S, generator=g, device=DEV))
        mix.out_proj.weight.copy_(torch.randn(8, S, generator=g, device=DEV))
        for name in ("q_proj", "k_proj", "v_proj", "out_proj"):
            setattr(mix, name, Int8Linear.from_float(getattr(mix, name)).eval())
        y = mix(x)
        bits = R.pack_bits3(*mix._fused_projections(x))
        sign, _ = R.match_packed(*(b.reshape(S, -1) for b in bits), 3)
        hard = mix.payload[None, :, None] * sign.reshape(1, S, 3).float()
        assert torch.equal(y, mix.out_proj(hard.permute(0, 2, 1).to(x.dtype)))
