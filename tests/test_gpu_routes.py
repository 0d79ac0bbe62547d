"""Per-query and turn routes against each other where their work splits.

The full-sequence read routes every query (bitmask selections); a stream of
route period 1 routes every token as a turn of its own (ids in score order).
Both read the same fines at every position, so their outputs agree to the
bf16 rounding of the two reads (each within about 4e-3 of exact arithmetic),
while one wrong selection moves its query's heads by a tenth or more.
"""
import pytest
import torch

from oracle import tao_oracle as O
from tao_attention import (TaoConfig, new_state, tao_attention, tao_attention_decode,
                           tao_attention_prefill, training)
from test_gpu_parity import inputs, run_oracle, to_dev, run_hip, compare_snapshots, TOL

pytestmark = pytest.mark.gpu


def _tokens(tokens, heads, width, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    xs = [torch.randn(1, tokens, heads, width, generator=g, device="cuda").to(torch.bfloat16)
          for _ in range(5)]
    return xs, [torch.randn(heads, width, 3, generator=g, device="cuda") * 0.02 for _ in range(2)]


@pytest.mark.parametrize("tokens,heads,width", [
    (769, 1, 64),          # one query with history, in a tile of one
    (1057, 2, 128),        # a ragged second tile: slots of one workgroup in two epochs
    (2337, 3, 64),         # seven fines, the last read tile holds one query
    (9001, 2, 128),        # chosen pages below all pages
    (9001, 1, 128),        # eight waves a workgroup
    (5003, 6, 128),        # two read tiles a workgroup
    (9001, 5, 64),         # the same
    (17000, 1, 64),        # more than 64 fines: selection keys stay in LDS; eight waves
    (262900, 1, 128),      # 1024 fines: one read tile per workgroup
])
def test_query_routes_equal_single_turn_routes(device, tokens, heads, width):
    print(f"routes T={tokens} H={heads} D={width}", flush=True)
    (q, k, v, rq, rk), (fa, fb) = _tokens(tokens, heads, width, tokens)
    named = dict(fusion_a=fa, fusion_b=fb, alpha=0.5)
    full, qsel = training.forward(q, k, v, rq, rk, fa, fb, 0.5, TaoConfig(coarse_index_only=True),
                                  return_routes=True)
    tail = min(tokens, 900)
    state = new_state(0, TaoConfig(coarse_index_only=True, route_period=1))
    if tokens > tail:
        state._ingest(*(x[:, :tokens - tail].contiguous() for x in (q, k, v, rq, rk)))
    cut = [x[:, tokens - tail:].contiguous() for x in (q, k, v, rq, rk)]
    out, state = tao_attention_prefill(*cut[:3], raw_q=cut[3], raw_k=cut[4], state=state,
                                       position=state.get_pos(), **named)
    a, b = full[:, tokens - tail:].double(), out.double()
    rows = (a - b).norm(dim=-1) / a.norm(dim=-1)
    assert rows.max().item() < 0.03
    words = qsel[0, tokens - 1]                                   # [H, W]
    picked = state.export()["route_ids"][1][0, 0]                 # [H, M] in score order
    for h in range(heads):
        bits = [f for f in range(32 * words.shape[-1])
                if (words[h, f // 32].item() >> (f % 32)) & 1]
        assert sorted(picked[h].tolist()) == bits


@pytest.mark.parametrize("period,layer", [(5, 0), (24, 3), (256, 1), (300, 0)])
def test_turn_routes_of_any_period_match_the_oracle(device, period, layer):
    """More than sixteen turns in an epoch, epochs without a turn, and the
    first turn of a staggered layer: route ids exact, outputs to tolerance."""
    config = TaoConfig(coarse_index_only=True, route_period=period)
    xs, fa, fb = inputs(4500, 2, 64, seed=period)
    splits = [2500, 1, 1999]
    state = new_state(layer, config)
    out = run_hip(state, to_dev(xs, device), fa.to(device), fb.to(device), splits)
    ora, ref = run_oracle(layer, xs, fa, fb, splits, geometry=O.Geometry.from_config(config))
    torch.testing.assert_close(out.cpu().float(), ref.float(), **TOL)
    compare_snapshots(state.export(), ora.export())


@pytest.mark.parametrize("width", [64, 128])
def test_turn_routes_near_two_thousand_fines(device, width):
    """A prompt chunk at 2,044 and 2,045 visible fines: its last turn routes
    as a decode step's refresh at the same token does (another kernel, the same
    arithmetic), bit for bit; the heads differ by the bf16 rounding of the two
    reads (about 4e-3 each)."""
    print(f"turn routes near 2,048 fines D={width}", flush=True)
    turn = 524280                                  # 768 + 24 k
    (q, k, v, rq, rk), (fa, fb) = _tokens(turn + 1, 1, width, width)
    xs = (q, k, v, rq, rk)
    named = dict(fusion_a=fa, fusion_b=fb, alpha=0.5)
    outs, routes = [], []
    for cut, call in ((turn - 300, tao_attention_prefill), (turn, tao_attention_decode)):
        state = new_state(0, TaoConfig(coarse_index_only=True))
        state._ingest(*(x[:, :cut].contiguous() for x in xs))
        c = [x[:, cut:].contiguous() for x in xs]
        out, state = call(*c[:3], raw_q=c[3], raw_k=c[4], state=state, position=cut, **named)
        outs.append(out[:, -1].double())
        routes.append(state.export()["route_ids"])
        del state
    for a, b in zip(*routes):
        assert torch.equal(a, b)
    assert ((outs[0] - outs[1]).norm() / outs[1].norm()).item() < 0.03
