"""The host-side facts of a step (core/attention_hip.py): kept for its layers, never past
a change of its lengths."""

from __future__ import annotations

import pytest
import torch

from inference_server.core import attention_hip
from inference_server.core.attention_hip import attach_host, paged_attention_hip_launch
from oracle.gather import paged_attention_gather as oracle_gather


class _Lengths:
    """A stand-in for device lengths with a host copy attached (no GPU needed)."""

    def __init__(self, values):
        self.device = torch.device("meta")
        self._pkv_host = torch.tensor(values)


def test_facts_are_shared_until_the_lengths_change():
    ctx, ql = _Lengths([20, 33]), _Lengths([4, 1])
    first = attention_hip._batch_facts(ctx, ql, 16, 4)
    assert attention_hip._batch_facts(ctx, ql, 16, 4) is first
    assert attention_hip._batch_facts(ctx, ql, 16, 2) is not first      # another table width
    assert attention_hip._batch_facts(ctx, ql, 16, 2)["too_few_blocks"]
    ql._pkv_host[1] = 2                                                  # in place, same tensor
    changed = attention_hip._batch_facts(ctx, ql, 16, 4)
    assert changed["total"] == 6 and changed["max_q"] == 4 and changed["qsl"] == {}
    ctx._pkv_host = torch.tensor([20, 65])                               # attached anew
    assert attention_hip._batch_facts(ctx, ql, 16, 4)["too_few_blocks"]


def test_kept_lengths_are_not_the_callers_tensors():
    """A host tensor of another step's values must not show through facts that an equal one
    attached since still finds."""
    hctx, hql = torch.tensor([20, 33]), torch.tensor([4, 1])
    ctx, ql = _Lengths([20, 33]), _Lengths([4, 1])
    ctx._pkv_host, ql._pkv_host = hctx, hql
    first = attention_hip._batch_facts(ctx, ql, 16, 4)
    ctx._pkv_host, ql._pkv_host = hctx.clone(), hql.clone()
    hctx.copy_(torch.tensor([64, 1]))
    hql.copy_(torch.tensor([1, 1]))
    assert attention_hip._batch_facts(ctx, ql, 16, 4) is first
    assert first["hctx"].tolist() == [20, 33] and first["hql"].tolist() == [4, 1]


@pytest.mark.gpu
def test_query_starts_follow_lengths_and_streams():
    """One upload per step and stream; lengths written in place make a new one (the same
    total and maximum, so nothing else would notice)."""
    g = torch.Generator().manual_seed(3)
    k, v = (torch.randn(16, 16, 2, 64, generator=g).half().cuda() for _ in range(2))
    tables = torch.arange(16).view(2, 8).cuda()
    q = torch.randn(9, 4, 64, generator=g).half().cuda()
    hctx, hql = torch.tensor([90, 70]), torch.tensor([7, 2])
    ctx, ql = attach_host(hctx.cuda(), hctx), attach_host(hql.cuda(), hql)

    def check():
        out = paged_attention_hip_launch(q, k, v, tables, ctx, ql, 0.125)
        ref = oracle_gather(q.cpu(), k.cpu(), v.cpu(), tables.cpu(), hctx, hql, 0.125)
        torch.testing.assert_close(out.cpu(), ref, atol=2e-2, rtol=2e-2)

    check()
    check()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        check()
    torch.cuda.current_stream().wait_stream(side)
    hql.copy_(torch.tensor([2, 7]))
    ql.copy_(hql)
    check()


@pytest.mark.gpu
def test_a_warmed_prefill_call_can_be_captured():
    """With host lengths attached and one call before the capture, the graph reads the
    query_start_loc of that call, which outlives a change of the lengths' facts."""
    g = torch.Generator().manual_seed(4)
    k, v = (torch.randn(16, 16, 2, 64, generator=g).half().cuda() for _ in range(2))
    tables = torch.arange(16).view(2, 8).cuda()
    q = torch.randn(9, 4, 64, generator=g).half().cuda()
    hctx, hql = torch.tensor([90, 70]), torch.tensor([7, 2])
    ctx, ql = attach_host(hctx.cuda(), hctx.clone()), attach_host(hql.cuda(), hql.clone())
    call = lambda: paged_attention_hip_launch(q, k, v, tables, ctx, ql, 0.125)  # noqa: E731
    eager = call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    # Other lengths through the same tensors' facts, and their memory handed out again.
    attach_host(ql, torch.tensor([2, 7]))
    call()
    del call
    spare = [torch.full((3,), -1, dtype=torch.long, device="cuda") for _ in range(64)]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    del spare
