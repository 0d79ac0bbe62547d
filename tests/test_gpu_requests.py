"""Requests issued one after another without waiting for the GPU: a finished
request's state is freed in its stream's order while its kernels still run."""
import pytest
import torch

from tao_attention import (TaoConfig, new_state, tao_attention_decode, tao_attention_prefill)
from tao_attention.tao_stream import DecodeBatch

pytestmark = pytest.mark.gpu


def _request(xs, fusion, config, steps):
    state, outs = new_state(0, config), []
    cuts = [(0, xs[0].shape[1] - steps)] + [(i, 1) for i in range(xs[0].shape[1] - steps,
                                                                  xs[0].shape[1])]
    for at, n in cuts:
        q, k, v, rq, rk = (x[:, at:at + n].contiguous() for x in xs)
        call = tao_attention_prefill if n > 1 else tao_attention_decode
        out, state = call(q, k, v, raw_q=rq, raw_k=rk, fusion_a=fusion[0], fusion_b=fusion[1],
                          alpha=0.5, state=state, position=state.get_pos())
        outs.append(out)
    return torch.cat(outs, 1), state


@pytest.mark.parametrize("side_stream", [False, True])
def test_requests_in_flight_do_not_share_memory(device, side_stream):
    g = torch.Generator(device=device).manual_seed(9)
    config = TaoConfig()
    fusion = [torch.randn(4, 128, 3, generator=g, device=device) * 0.02 for _ in range(2)]
    inputs = [[torch.randn(1, n, 4, 128, generator=g, device=device).to(torch.bfloat16)
               for _ in range(5)] for n in (2900, 1100, 3300)]
    want = []
    for xs in inputs:
        want.append(_request(xs, fusion, config, 3)[0])
        torch.cuda.synchronize()
    stream = torch.cuda.Stream() if side_stream else torch.cuda.current_stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        got = [_request(inputs[i % 3], fusion, config, 3)[0] for i in range(12)]
    torch.cuda.synchronize()
    for i, out in enumerate(got):
        assert torch.equal(out, want[i % 3])


@pytest.mark.parametrize("inside", [True, False])
@pytest.mark.parametrize("steps", [1, 3])
def test_a_state_used_on_another_stream_is_drained(device, inside, steps):
    """Buffers of the default stream, decodes on a side stream behind work
    that takes its time: closing the driver waits for the side stream before
    the buffers are freed, whichever stream is current where the state goes."""
    g = torch.Generator(device=device).manual_seed(10)
    fusion = [torch.randn(2, 64, 3, generator=g, device=device) * 0.02 for _ in range(2)]
    xs = [torch.randn(1, 800 + steps, 2, 64, generator=g, device=device).to(torch.bfloat16)
          for _ in range(5)]
    _, state = _request([x[:, :800] for x in xs], fusion, TaoConfig(), 1)
    assert not state._drain
    big = torch.randn(8192, 8192, generator=g, device=device)
    big @ big                                      # the library's own first call
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    cuts = [[x[:, i:i + 1].contiguous() for x in xs] for i in range(800, 800 + steps)]
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):
            busy = big @ big
        for q, k, v, rq, rk in cuts:
            _, state = tao_attention_decode(q, k, v, raw_q=rq, raw_k=rk, fusion_a=fusion[0],
                                            fusion_b=fusion[1], alpha=0.5, state=state,
                                            position=state.get_pos())
        assert state._drain and not side.query()
        if inside:
            del state
            assert side.query()
    if not inside:
        del state
        assert side.query()
    del busy


@pytest.mark.parametrize("states_first", [True, False])
def test_a_batch_used_on_another_stream_is_drained(device, states_first):
    """A batch opened on the default stream and stepped on a side stream: its
    table and its states' buffers go after the side stream's work."""
    g = torch.Generator(device=device).manual_seed(11)
    fusion = [torch.randn(2, 64, 3, generator=g, device=device) * 0.02 for _ in range(2)]
    xs = [torch.randn(2, 802, 2, 64, generator=g, device=device).to(torch.bfloat16)
          for _ in range(5)]
    states = [_request([x[r:r + 1, :800].contiguous() for x in xs], fusion, TaoConfig(), 1)[1]
              for r in range(2)]
    batch = DecodeBatch(states)
    first, second = ([x[:, i:i + 1].contiguous() for x in xs] for i in (800, 801))
    batch.decode(*first, *fusion, 0.5)
    big = torch.randn(8192, 8192, generator=g, device=device)
    big @ big                                      # the library's own first call
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):
            busy = big @ big
        batch.decode(*second, *fusion, 0.5)
        assert not side.query()
    if states_first:
        batch.states = []
        del states                                 # each waits for the side stream
        assert side.query()
    else:
        batch.close()                              # the table's own wait
        assert side.query()
    del busy


def test_growth_on_another_stream_waits_for_the_old_buffers(device):
    """A prompt chunk on a side stream that outgrows a state's bank: the old
    buffers are the default stream's, and are still read behind work that takes
    its time. The outputs are those of one stream."""
    g = torch.Generator(device=device).manual_seed(12)
    fusion = [torch.randn(2, 64, 3, generator=g, device=device) * 0.02 for _ in range(2)]
    xs = [torch.randn(1, 6000, 2, 64, generator=g, device=device).to(torch.bfloat16)
          for _ in range(5)]
    named = dict(fusion_a=fusion[0], fusion_b=fusion[1], alpha=0.5)
    big = torch.randn(8192, 8192, generator=g, device=device)
    big @ big                                      # the library's own first call
    outs = []
    for stream in (torch.cuda.current_stream(), torch.cuda.Stream()):
        state = new_state(0, TaoConfig())
        for lo, hi, at in ((0, 1500, torch.cuda.current_stream()), (1500, 6000, stream)):
            q, k, v, rq, rk = (x[:, lo:hi].contiguous() for x in xs)
            torch.cuda.synchronize()
            with torch.cuda.stream(at):
                if lo:
                    for _ in range(20):
                        busy = big @ big
                before = torch.cuda.Event()
                before.record()
                out, state = tao_attention_prefill(q, k, v, raw_q=rq, raw_k=rk, state=state,
                                                   position=state.get_pos(), **named)
        if state._drain:
            assert before.query()
        torch.cuda.synchronize()
        outs.append(out)
    assert state._drain and torch.equal(*outs)
    del busy
