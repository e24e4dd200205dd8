"""GPU parity of the causal GQA prefill attention core (ie_attn_prefill_core) against a plain
PyTorch fp32 reference of the same op, at prompt lengths up to BASELINE config 4's 2048 rows
and with a cached prefix (start_pos > 0).  Tolerance: tests/tolerance.py (max-abs / scale and
mean relative error <= 1e-2); the kernel rounds the probabilities to bf16 before P.V, as the
reference's fp16 softmax output does (softmax.cu:55-107).
"""
import math

import pytest
import torch

from gpu_util import P, say
from tolerance import assert_close

pytestmark = pytest.mark.gpu
CTX = 8192


def reference(q, k, v, start_pos):
    """q [S][32][128], k/v [8][CTX][128] (bf16 tensors) -> [S][32][128] fp32."""
    S = q.shape[0]
    n = start_pos + S
    out = torch.empty(S, 32, 128, dtype=torch.float32, device="cuda")
    pos = torch.arange(S, device="cuda")[:, None] + start_pos
    keys = torch.arange(n, device="cuda")[None, :]
    masked = keys > pos
    for h in range(32):
        qh = q[:, h].float()
        kh = k[h // 4, :n].float()
        vh = v[h // 4, :n].float()
        s = torch.matmul(qh, kh.t().contiguous()) / math.sqrt(128.0)
        s = s.masked_fill(masked, float("-inf"))
        out[:, h] = torch.matmul(torch.softmax(s, dim=-1), vh)
    return out


# the kernel forms: 16 rows per 4-wave workgroup below 1280 rows, two 16-row blocks per 8-wave
# workgroup up to 2559 (1500 + 37: the two blocks of a workgroup end in different key tiles), 32
# rows per wave from 2560
@pytest.mark.parametrize("S,start_pos", [(1, 0), (17, 0), (96, 0), (300, 5), (1000, 0),
                                         (1500, 37), (2048, 0), (200, 2000), (2600, 0),
                                         (3000, 1000)])
def test_attn_prefill_core(hip, ctx, S, start_pos):
    say(f"attn_prefill_core S={S} start_pos={start_pos}")
    g = torch.Generator(device="cuda").manual_seed(1000 + S + start_pos)
    q = torch.randn(S, 32, 128, generator=g, device="cuda").to(torch.bfloat16)
    k = torch.zeros(8, CTX, 128, dtype=torch.bfloat16, device="cuda")
    v = torch.zeros_like(k)
    n = start_pos + S
    k[:, :n] = torch.randn(8, n, 128, generator=g, device="cuda").to(torch.bfloat16)
    v[:, :n] = torch.randn(8, n, 128, generator=g, device="cuda").to(torch.bfloat16)
    # rows past the context hold large finite values: the kernel must not read them
    k[:, n:n + 64] = 3.0e4
    v[:, n:n + 64] = 3.0e4
    out = torch.empty(S, 32 * 128, dtype=torch.bfloat16, device="cuda")
    hip.check(hip.lib.ie_attn_prefill_core(ctx.handle, S, start_pos, P(q), P(k), P(v), P(out)))
    torch.cuda.synchronize()
    want = reference(q, k, v, start_pos)
    assert_close(out.float().view(S, 32, 128).cpu().numpy(), want.cpu().numpy(),
                 what=f"attn prefill core S={S} start={start_pos}")


# key splits (few rows over many keys): runs that end inside a row block's masked tiles (33 rows
# at 1990), a run of one ragged tile, an empty last run (16 tiles in 7 runs of 3), one row, rows
# that do not fill a 16-row block, and the 4096 rows x splits limit (1300 x 3)
@pytest.mark.parametrize("S,start_pos", [(1, 1000), (1, 8191), (16, 1000), (33, 1990),
                                         (64, 4001), (200, 7992), (700, 7000), (1300, 6800)])
def test_attn_prefill_core_key_splits(hip, ctx, S, start_pos):
    say(f"attn_prefill_core key splits S={S} start_pos={start_pos}")
    g = torch.Generator(device="cuda").manual_seed(2000 + S + start_pos)
    q = (2 * torch.randn(S, 32, 128, generator=g, device="cuda")).to(torch.bfloat16)
    k = torch.full((8, CTX, 128), 3.0e4, dtype=torch.bfloat16, device="cuda")
    v = torch.full_like(k, 3.0e4)   # rows past the context: must not be read
    n = start_pos + S
    k[:, :n] = torch.randn(8, n, 128, generator=g, device="cuda").to(torch.bfloat16)
    v[:, :n] = torch.randn(8, n, 128, generator=g, device="cuda").to(torch.bfloat16)
    out = torch.full((S + 1, 32 * 128), 7.0, dtype=torch.bfloat16, device="cuda")
    hip.check(hip.lib.ie_attn_prefill_core(ctx.handle, S, start_pos, P(q), P(k), P(v), P(out)))
    # the same keys in shuffled pages
    npg = (n + 63) // 64
    pool = torch.full((npg, 32, 2, 8, 64, 128), 3.0e4, dtype=torch.bfloat16, device="cuda")
    order = torch.randperm(npg, generator=g, device="cuda")
    for kv, plane in ((k, 0), (v, 1)):
        rows = torch.full((8, npg * 64, 128), 3.0e4, dtype=torch.bfloat16, device="cuda")
        rows[:, :n] = kv[:, :n]
        pool[order, 3, plane] = rows.view(8, npg, 64, 128).transpose(0, 1).contiguous()
    paged = torch.empty(S, 32 * 128, dtype=torch.bfloat16, device="cuda")
    hip.check(hip.lib.ie_attn_prefill_core_paged(ctx.handle, S, start_pos, P(q), P(pool), npg,
                                                 P(order.to(torch.int32)), 3, P(paged)))
    torch.cuda.synchronize()
    want = reference(q, k, v, start_pos)
    assert_close(out[:S].float().view(S, 32, 128).cpu().numpy(), want.cpu().numpy(),
                 what=f"attn key splits S={S} start={start_pos}")
    assert torch.equal(out[:S], paged)
    assert bool((out[S] == 7.0).all())


def test_attn_prefill_core_key_splits_captured(hip):
    """Key-split sizes recorded into a caller's graphs: a recorded call takes no scratch of the
    context and runs unsplit, before and after an eager call with splits alike.  The graphs replay
    one after the other, at once on two streams beside eager split calls, and after the context
    is gone."""
    from infengine_amd.engine import Context
    say("attn_prefill_core key splits captured")
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(1300, 32, 128, generator=g, device="cuda").to(torch.bfloat16)
    k = torch.randn(8, CTX, 128, generator=g, device="cuda").to(torch.bfloat16)
    v = torch.randn(8, CTX, 128, generator=g, device="cuda").to(torch.bfloat16)
    first, second, eager, big = (torch.empty(S, 32 * 128, dtype=torch.bfloat16, device="cuda")
                                 for S in (64, 64, 64, 1300))
    torch.cuda.synchronize()
    stream, other = torch.cuda.Stream(), torch.cuda.Stream()
    c = Context(0, stream, graph=False)

    def attend(S, start, out):
        hip.check(hip.lib.ie_attn_prefill_core(c.handle, S, start, P(q), P(k), P(v), P(out)))

    graphs = []
    for out in (first, second):  # before and after the scratch is there
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            attend(64, 4001, out)
        graphs.append(graph)
        attend(64, 4001, eager)
        torch.cuda.synchronize()
    want = reference(q[:64], k, v, 4001).cpu().numpy()
    assert_close(eager.float().view(64, 32, 128).cpu().numpy(), want, what="eager, split")
    graphs[0].replay()
    torch.cuda.synchronize()
    unsplit = first.clone()
    assert_close(unsplit.float().view(64, 32, 128).cpu().numpy(), want, what="captured, unsplit")
    assert not torch.equal(unsplit, eager)  # (another order of the sums: the eager call was split)
    split = eager.clone()
    for turn in range(4):
        first.zero_(), second.zero_(), eager.zero_()
        torch.cuda.synchronize()
        if turn < 3:
            attend(64, 4001, eager)
            attend(1300, 6800, big)
        else:
            c.close()
        for s, graph in zip((stream, other), graphs):
            with torch.cuda.stream(s):
                graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(first, unsplit) and torch.equal(second, unsplit)
        assert turn == 3 or torch.equal(eager, split)


def test_attn_prefill_core_key_splits_beside_a_capture(hip):
    """The first split call of a context, which allocates its scratch, while another stream is being
    captured: the call runs split, and the capture ends and replays."""
    from infengine_amd.engine import Context
    say("attn_prefill_core key splits beside a capture")
    g = torch.Generator(device="cuda").manual_seed(4)
    q = torch.randn(64, 32, 128, generator=g, device="cuda").to(torch.bfloat16)
    k = torch.randn(8, CTX, 128, generator=g, device="cuda").to(torch.bfloat16)
    v = torch.randn(8, CTX, 128, generator=g, device="cuda").to(torch.bfloat16)
    outs = [torch.empty(64, 32 * 128, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    mark = torch.zeros(8, device="cuda")
    torch.cuda.synchronize()
    work, captured = torch.cuda.Stream(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    contexts = [Context(0, work, graph=False) for _ in outs]
    with torch.cuda.graph(graph, stream=captured):
        mark += 1
        hip.check(hip.lib.ie_attn_prefill_core(contexts[0].handle, 64, 4001, P(q), P(k), P(v), P(outs[0])))
    hip.check(hip.lib.ie_attn_prefill_core(contexts[1].handle, 64, 4001, P(q), P(k), P(v), P(outs[1])))
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and mark.tolist() == [3.0] * 8
    for c in contexts:
        c.close()


@pytest.mark.parametrize("S,start_pos,split", [(33, 500, False), (200, 900, False), (256, 1000, False),
                                               (512, 2000, False), (16, 600, True), (200, 3000, True),
                                               (512, 5000, True)])
def test_attn_prefill_core_splits_where_they_pay(hip, S, start_pos, split):
    """Few keys run unsplit, where two kernels took 5-13% longer than the one (22.6 against 19.9 us
    at 256 rows over 1256 keys): the bits of a recorded call, which never splits, are the eager
    call's exactly then."""
    from infengine_amd.engine import Context
    say(f"attn_prefill_core split or not S={S} start_pos={start_pos}")
    g = torch.Generator(device="cuda").manual_seed(S + start_pos)
    q = (2 * torch.randn(S, 32, 128, generator=g, device="cuda")).to(torch.bfloat16)
    k, v = (torch.randn(8, CTX, 128, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    eager, recorded = (torch.empty(S, 32 * 128, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    c = Context(0, stream, graph=False)
    hip.check(hip.lib.ie_attn_prefill_core(c.handle, S, start_pos, P(q), P(k), P(v), P(eager)))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        hip.check(hip.lib.ie_attn_prefill_core(c.handle, S, start_pos, P(q), P(k), P(v), P(recorded)))
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(eager, recorded) != split
    c.close()
