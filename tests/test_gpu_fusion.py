"""The read tiles' fusion, two channels at a time: tiles with and without the
coarse branch, a ragged last tile, flat and saturated branch weights."""
import pytest
import torch

from oracle import tao_oracle as O
from tao_attention import TaoConfig, training

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [64, 128])
@pytest.mark.parametrize("scale,alpha", [(0.0, 0.5), (3.0, -1.25)])
def test_tile_fusion_matches_oracle(device, width, scale, alpha):
    """Every rounding point is the oracle's, so the logits agree exactly; the
    outputs differ by the reads' own orders (2e-2 relative, the bf16 bar) and
    by one bf16 step of each branch's weight and term."""
    g = torch.Generator().manual_seed(51 + width)
    tokens, heads = 2871, 2
    xs = [torch.randn(1, tokens, heads, width, generator=g).to(torch.bfloat16)
          for _ in range(5)]
    fa, fb = (torch.randn(heads, width, 3, generator=g) * scale for _ in range(2))
    cfg = TaoConfig()
    out = training.forward(*(x.to(device) for x in xs), fa.to(device), fb.to(device), alpha,
                           cfg).float().cpu()
    ref = O.training_forward(*xs, fa, fb, alpha, O.Geometry.from_config(cfg)).float()
    for lo, hi in ((0, 768), (768, 2560), (2560, tokens)):     # local; fine; coarse too
        err = (out[:, lo:hi] - ref[:, lo:hi]).norm() / ref[:, lo:hi].norm()
        assert err < 2e-2, (lo, float(err))
        top = ref[:, lo:hi].abs().max()
        assert (out[:, lo:hi] - ref[:, lo:hi]).abs().max() < 2e-2 * top
    assert torch.isfinite(out).all()
