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


@pytest.mark.parametrize("index_only", [False, True])
def test_heads_read_the_same_alone_and_among_many(device, index_only):
    """Two heads alone (a workgroup a CU) and among 28 (two a CU, another build
    of the read; two query tiles a routing workgroup): the same bits."""
    g = torch.Generator(device=device).manual_seed(61)
    tokens, heads, width = 2900, 28, 64
    xs = [torch.randn(1, tokens, heads, width, generator=g, device=device).to(torch.bfloat16)
          for _ in range(5)]
    fa, fb = (torch.randn(heads, width, 3, generator=g, device=device) * 0.02 for _ in range(2))
    cfg = TaoConfig(coarse_index_only=index_only)
    many = training.forward(*xs, fa, fb, 0.5, cfg)
    few = training.forward(*(x[:, :, :2].contiguous() for x in xs), fa[:2], fb[:2], 0.5, cfg)
    assert torch.equal(many[:, :, :2], few)
