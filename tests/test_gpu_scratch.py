"""Contexts that have no scratch to give: what an operator does then."""
import numpy as np
import pytest
import torch

from diopi_amd import functions as F
from diopi_amd import runtime as rt
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _captured(call, stream):
    """Records `call` on a new context whose pool is empty, so that every request for scratch meets a capture."""
    ctx = rt.Context(stream=stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call(ctx)
    assert ctx.malloc_count == 0
    return graph, ctx


def test_heads_of_64_are_captured_without_scratch():
    """Heads of 64 can do without: one range for a sequence, the general attention kernel in the place of the one that takes a plan."""
    g = torch.Generator().manual_seed(41)
    rand = lambda *shape: torch.randn(*shape, generator=g).half().to(DEV)
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    lens = [3000, 700, 5]
    total, longest = sum(lens), max(lens)
    table = torch.zeros(3, longest, dtype=torch.int32)
    start = np.concatenate(([0], np.cumsum(lens)))[:-1].tolist()
    for i, n in enumerate(lens):
        table[i, longest - n:] = torch.arange(start[i], start[i] + n)
    logits, cache, out = rand(8, total), rand(total, 2, 64), torch.zeros(3, 8, 64, dtype=torch.float16, device=DEV)
    tables = (table.to(DEV), ints(start), ints(lens))
    decode = lambda ctx=None: F.token_softmax_reducev(logits, cache, out, *tables, longest, 0, ctx=ctx)
    many = [5 + i % 9 for i in range(70)]  # more sequences than a wave has lanes: their tiles come from a table
    q, k, v = (rand(sum(many), 2, 64) for _ in range(3))
    loc, length, att = ints(np.concatenate(([0], np.cumsum(many)))[:-1].tolist()), ints(many), torch.zeros_like(q)
    attend = lambda ctx=None: F.context_attention(q, k, v, att, loc, length, max(many), ctx=ctx)
    for call, result, value in ((decode, out, cache), (attend, att, v)):
        stream = torch.cuda.Stream()
        graph, ctx = _captured(call, stream)
        for _ in range(3):
            value.copy_(torch.randn(value.shape, generator=g))
            result.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            got = result.clone()
            call()
            torch.cuda.synchronize()
            assert_close(got, result, rtol=4 * 2.0 ** -11, atol=2.0 ** -9, what="a replay without scratch")
        del graph
        ctx.close()


def test_a_refused_call_leaves_a_capture_valid():
    """Heads of 128 need their scratch: the call fails, and the graph goes on without it."""
    stream = torch.cuda.Stream()
    v = torch.randn(4, 1, 128).half().to(DEV)
    logits, out = torch.zeros(1, 4, dtype=torch.float16, device=DEV), torch.zeros(1, 1, 128, dtype=torch.float16, device=DEV)
    table, start, length = torch.zeros(1, 5000, dtype=torch.int32, device=DEV), *(torch.tensor([x], dtype=torch.int32, device=DEV) for x in (0, 4))
    x = torch.ones(8, device=DEV)
    ctx, graph = rt.Context(stream=stream), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        with pytest.raises(rt.DiopiException, match="failed"):
            F.token_softmax_reducev(logits, v, out, table, start, length, 5000, 0, ctx=ctx)
        y = x + 1
    x.fill_(3)
    graph.replay()
    torch.cuda.synchronize()
    assert (y == 4).all()
    F.token_softmax_reducev(logits, v, out, table, start, length, 5000, 0, ctx=ctx)
    torch.cuda.synchronize()
    assert_close(out[0, 0], v[0, 0], rtol=2.0 ** -10, atol=2.0 ** -24, what="the same call outside")
    ctx.close()


def test_memory_that_the_device_does_not_have():
    """The call that asked for it fails; the next one is not held responsible."""
    ctx = rt.Context()
    window, H = 65535 * 2048, 16384  # 558 GB of partial sums
    v = torch.randn(4, H, 128).half().to(DEV)
    logits, out = torch.zeros(H, 4, dtype=torch.float16, device=DEV), torch.zeros(1, H, 128, dtype=torch.float16, device=DEV)
    table, start, length = torch.zeros(1, window, dtype=torch.int32, device=DEV), *(torch.tensor([x], dtype=torch.int32, device=DEV) for x in (0, 4))
    for c in (ctx, None):
        with pytest.raises(rt.DiopiException, match="failed"):
            F.token_softmax_reducev(logits, v, out, table, start, length, window, 0, ctx=c)
        F.token_softmax_reducev(logits, v, out, table, start, length, 2048, 0, ctx=c)
        torch.cuda.synchronize()
        assert_close(out[0], v[0], rtol=2.0 ** -10, atol=2.0 ** -24, what="the next call")
    ctx.close()
