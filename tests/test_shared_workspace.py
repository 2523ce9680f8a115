"""Calls of different kernels on one workspace: what one leaves behind is what the next relies
on (the merge counters at its front must read zero when a split decode starts)."""

from __future__ import annotations

import pytest
import torch

from inference_server import native
from inference_server.core.attention_hip import _WORKSPACES, attach_host, paged_attention_hip_launch
from oracle.gather import paged_attention_gather as oracle_gather

pytestmark = pytest.mark.gpu


def _batch(ctx, *, kv, group, d, seed):
    g = torch.Generator().manual_seed(seed)
    n, width = len(ctx), -(-max(ctx) // 16)
    rand = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    # Sequences share blocks: attention only reads them.
    blocks = width + 3
    tables = torch.stack([torch.randperm(blocks, generator=g)[:width] for _ in range(n)])
    return (rand(n, kv * group, d), rand(blocks, 16, kv, d), rand(blocks, 16, kv, d), tables, torch.tensor(ctx),
            torch.ones(n, dtype=torch.long))


#: The shortest contexts the persistent kernel takes (512 sequences of 8 KV heads x 128), none
#: longer than one split-KV partial, and contexts that the one-launch kernel splits.
def _persistent():
    return _batch([256] * 500 + [1 + 21 * i for i in range(12)], kv=8, group=4, d=128, seed=1)


def _split():
    return _batch([3000, 40, 1900, 700], kv=8, group=4, d=128, seed=2)


def _check(b, out, rows):
    q, k, v, tables, ctx, ql = b
    ref = oracle_gather(q[rows], k, v, tables[rows], ctx[rows], ql[rows], 128 ** -0.5)
    torch.testing.assert_close(out.cpu()[rows], ref, atol=2e-2, rtol=2e-2)


def test_split_decode_after_a_persistent_batch_of_short_contexts():
    for b, rows in ((_split(), [0, 1, 2, 3]), (_persistent(), [0, 499, 500, 511]), (_split(), [0, 1, 2, 3]),
                    (_split(), [0, 1, 2, 3])):
        out = paged_attention_hip_launch(*(t.cuda() for t in b), 128 ** -0.5)
        torch.cuda.synchronize()
        _check(b, out, rows)
    stream = torch.cuda.current_stream().cuda_stream
    ws = _WORKSPACES.partials(torch.device("cuda", 0), stream, 1)
    assert int(ws[:256 * 1024].count_nonzero()) == 0


def test_the_same_on_the_static_scratch():
    L = native.lib()
    for b, rows in ((_persistent(), [0, 499, 500, 511]), (_split(), [0, 1, 2, 3]), (_split(), [0, 1, 2, 3])):
        q, k, v, tables, ctx, _ = (t.cuda() for t in b)
        out = torch.full_like(q, float("nan"))
        rc = L.pkv_paged_attention_decode_noalloc(
            out.data_ptr(), out.stride(0), out.stride(1), q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(),
            v.data_ptr(), *k.stride()[:3], *k.shape, tables.data_ptr(), tables.stride(0), tables.shape[1],
            ctx.data_ptr(), q.shape[0], q.shape[1], int(b[4].max()), 128 ** -0.5, native.PKV_BFLOAT16,
            torch.cuda.current_stream().cuda_stream)
        native.check(rc, "pkv_paged_attention_decode_noalloc")
        torch.cuda.synchronize()
        _check(b, out, rows)


def test_a_capture_clears_one_workspace_for_all_its_calls():
    """Captures on a stream without a workspace: one fill node each, whatever the calls, and
    each capture its own (the second one is replayed first)."""
    from inference_server.core.decode_graphs import node_census

    b = [t.cuda() for t in _split()]
    hosts = (_split()[4], _split()[5])
    attach_host(b[4], hosts[0])
    attach_host(b[5], hosts[1])
    eager = paged_attention_hip_launch(*b, 128 ** -0.5)
    stream, graphs = torch.cuda.Stream(), []
    for _ in range(2):
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph, stream=stream):
            outs = [paged_attention_hip_launch(*b, 128 ** -0.5) for _ in range(3)]
        assert node_census(graph) == {"kernel": 3 + 1}
        graph.instantiate()
        graphs.append((graph, outs))
    for _ in range(2):
        for graph, outs in reversed(graphs):
            for o in outs:
                o.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(o, eager) for o in outs)
