"""The one-launch MFMA decode kernel (csrc/attn_decode_split.hip) against oracle.gather at the
bars of 2e-2 in 16 bits and 1e-5 in fp32: head_dims, groups, block sizes, contexts around the edges of a unit (16
keys), a wave's round (4 or 8 units) and a run, sequence counts around the 64 lanes and 16
sequences per lane of its run search, runs longer than the 32 units whose block ids a wave
holds, and the fused append. Pool rows no key may come from are NaN.
"""

from __future__ import annotations

import pytest
import torch

from inference_server import native
from inference_server.core.attention_hip import attach_host, paged_attention_hip_launch
from inference_server.core.decode_graphs import capture_step
from oracle.gather import paged_attention_gather as oracle_gather

pytestmark = pytest.mark.gpu
TOL = {torch.float16: 2e-2, torch.bfloat16: 2e-2, torch.float32: 1e-5}


def _batch(ctx, *, dtype, d, bs, kv, group, seed=0):
    g = torch.Generator().manual_seed(seed)
    need = [-(-c // bs) for c in ctx]
    num_blocks = sum(need) + 2
    perm = torch.randperm(num_blocks, generator=g).tolist()
    tables = torch.zeros(len(ctx), max(need) + 1, dtype=torch.long)
    live = torch.zeros(num_blocks, bs, dtype=torch.bool)
    at = 0
    for i, (c, n) in enumerate(zip(ctx, need)):
        tables[i, :n] = torch.tensor(perm[at:at + n])
        at += n
        pos = torch.arange(c)
        live[tables[i, pos // bs], pos % bs] = True
    rand = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    k, v = rand(num_blocks, bs, kv, d), rand(num_blocks, bs, kv, d)
    k[~live], v[~live] = float("nan"), float("nan")
    n = len(ctx)
    return dict(q=2 * rand(n, kv * group, d), k=k, v=v, tables=tables, ctx=torch.tensor(ctx),
                k_new=rand(n, kv, d), v_new=rand(n, kv, d))


def _run(b, *, fused):
    n, bs, d = len(b["ctx"]), b["k"].shape[1], b["q"].shape[2]
    last = b["ctx"] - 1
    slots = b["tables"][torch.arange(n), last // bs] * bs + last % bs
    k, v = b["k"].clone(), b["v"].clone()
    if fused:                                   # what the call must not read: the new slots
        k.view(-1, *k.shape[2:])[slots] = float("nan")
        v.view(-1, *v.shape[2:])[slots] = float("nan")
    kd, vd = k.cuda(), v.cuda()
    append = (b["k_new"].cuda(), b["v_new"].cuda(), slots.cuda()) if fused else None
    args = (b["q"].cuda(), kd, vd, b["tables"].cuda(), b["ctx"].cuda(), torch.ones(n, dtype=torch.long).cuda(), d ** -0.5)
    outs = [paged_attention_hip_launch(*args, append=append) for _ in range(2)]
    torch.cuda.synchronize()
    if fused:
        k.view(-1, *k.shape[2:])[slots] = b["k_new"]
        v.view(-1, *v.shape[2:])[slots] = b["v_new"]
    bits = lambda t: t.cpu().view(torch.int32 if t.dtype == torch.float32 else torch.int16)  # noqa: E731
    assert torch.equal(bits(kd), bits(k)) and torch.equal(bits(vd), bits(v))
    assert torch.equal(bits(outs[0]), bits(outs[1]))        # and the merge counters were left zero
    return outs[0].cpu(), k, v, slots


def _check(b, *, fused, rows=None):
    out, k, v, _ = _run(b, fused=fused)
    rows = torch.arange(len(b["ctx"])) if rows is None else torch.tensor(rows)
    clean = lambda t: torch.nan_to_num(t)  # noqa: E731  (never read: the oracle masks, 0 x NaN is NaN)
    ref = oracle_gather(b["q"][rows], clean(k), clean(v), b["tables"][rows], b["ctx"][rows],
                        torch.ones(len(rows), dtype=torch.long), b["q"].shape[2] ** -0.5)
    torch.testing.assert_close(out[rows], ref, atol=TOL[out.dtype], rtol=TOL[out.dtype])


EDGES = [1, 7, 8, 9, 15, 16, 17, 63, 64, 65, 127, 129, 512, 513]


@pytest.mark.parametrize("d,bs,kv,group,dtype", [
    (32, 8, 2, 16, torch.float16), (32, 16, 3, 1, torch.bfloat16), (48, 16, 1, 5, torch.bfloat16),
    (64, 16, 12, 1, torch.float16), (64, 32, 3, 7, torch.bfloat16), (80, 8, 2, 2, torch.float16),
    (80, 16, 1, 12, torch.bfloat16), (96, 64, 2, 3, torch.float16), (112, 16, 1, 4, torch.bfloat16),
    (128, 16, 8, 4, torch.bfloat16), (128, 8, 1, 8, torch.float16), (128, 128, 2, 9, torch.float16),
    (32, 8, 2, 3, torch.float32), (48, 32, 1, 16, torch.float32), (64, 16, 12, 1, torch.float32),
    (80, 8, 2, 2, torch.float32), (112, 16, 1, 5, torch.float32), (128, 16, 2, 4, torch.float32)])
@pytest.mark.parametrize("fused", [False, True], ids=["plain", "append"])
def test_shapes_and_context_edges(d, bs, kv, group, dtype, fused):
    _check(_batch(EDGES, dtype=dtype, d=d, bs=bs, kv=kv, group=group, seed=d + bs), fused=fused)


@pytest.mark.parametrize("n,dtype", [(n, torch.bfloat16) for n in (1, 2, 63, 64, 65, 130, 300)]
                         + [(n, torch.float32) for n in (2, 66)])
@pytest.mark.parametrize("fused", [False, True], ids=["plain", "append"])
def test_run_search_over_sequence_counts(n, dtype, fused):
    """Long contexts among short ones, so that runs are cut and found across lanes."""
    ctx = [5 + (37 * i) % 150 for i in range(n)]
    for i, c in ((0, 3000), (n // 2, 1900), (n - 1, 4099)):
        ctx[i] = c
    rows = sorted({0, n // 2, n - 1, n // 3, max(0, n - 2)})
    _check(_batch(ctx, dtype=dtype, d=64, bs=16, kv=1, group=4, seed=n), fused=fused, rows=rows)


@pytest.mark.parametrize("n,kv,d,long", [
    (350, 3, 32, 2200),      # more pairs than the GPU holds, long contexts: runs for two rounds
    (350, 3, 32, 1300),      # the same, none long enough: unsplit
    (1030, 1, 64, 300),      # more sequences than the search takes
    (1100, 1, 64, 5000),     # the same, with contexts that would outlast the others
    (600, 2, 128, 8192),     # two rounds of pairs, likewise
    (700, 6, 64, 90),        # many rounds of pairs: two waves a workgroup
    (40, 3, 128, 9000)],     # a few long contexts, cut into short runs
    ids=["two rounds", "unsplit", "many", "many, outliers", "outliers", "rounds", "long"])
def test_unsplit_and_long_runs(n, kv, d, long):
    ctx = [1 + (29 * i) % 70 for i in range(n)]
    ctx[1], ctx[n // 2], ctx[n - 1] = long, long - 7, long + 13
    _check(_batch(ctx, dtype=torch.float16, d=d, bs=16, kv=kv, group=2, seed=n + d), fused=True,
           rows=[0, 1, 2, n // 2, n - 2, n - 1])


@pytest.mark.parametrize("n,ctx,dtype,kv,group,d,bs", [
    (8, 42000, torch.float16, 8, 1, 64, 16),         # runs of ~44 units a wave
    (6, 50000, torch.bfloat16, 4, 2, 80, 32),        # ~38
    (6, 60000, torch.float32, 2, 4, 128, 16),        # ~45
    (1030, 4800, torch.float16, 1, 2, 64, 8)],       # past the search, none outlying: 75, uncut
    ids=["fp16", "bf16", "fp32", "uncut"])
@pytest.mark.parametrize("fused", [False, True], ids=["plain", "append"])
def test_waves_of_more_units_than_they_hold_block_ids_of(n, ctx, dtype, kv, group, d, bs, fused):
    """A wave holds the block ids of 32 units: these take the next ones and start their ring
    anew. Sequences share blocks, but for the one that holds their new token."""
    g = torch.Generator().manual_seed(n)
    ctxs = [ctx + (13 * i) % 97 for i in range(n)]
    need = [-(-c // bs) for c in ctxs]
    shared = 600
    tables = torch.randint(0, shared, (n, max(need) + 1), generator=g)
    tables[torch.arange(n), torch.tensor(need) - 1] = shared + torch.randperm(n, generator=g)
    rand = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    b = dict(q=2 * rand(n, kv * group, d), k=rand(shared + n, bs, kv, d), v=rand(shared + n, bs, kv, d), tables=tables,
             ctx=torch.tensor(ctxs), k_new=rand(n, kv, d), v_new=rand(n, kv, d))
    _check(b, fused=fused, rows=[0, n // 2, n - 1])


def test_contexts_of_zero_write_nothing_and_split_nothing():
    b = _batch([2500, 40, 17], dtype=torch.float16, d=128, bs=16, kv=2, group=4, seed=5)
    ref, _, _, _ = _run(b, fused=False)
    L, dev, s = native.lib(), "cuda", torch.cuda.current_stream().cuda_stream
    tables = torch.cat([b["tables"][:1], torch.zeros_like(b["tables"][:1]), b["tables"][1:]]).to(dev)
    ctx = torch.tensor([2500, 0, 40, 17], device=dev)
    q = torch.cat([b["q"][:1], b["q"][:1], b["q"][1:]]).to(dev)
    k, v = b["k"].to(dev), b["v"].to(dev)
    out = torch.full((4, 8, 129), 7.0, dtype=torch.float16, device=dev)[:, :, :128]    # rows of 129: 2-byte stores
    need = L.pkv_paged_attention_decode_workspace_bytes(4, 8, 2, 128, 2500)
    ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    rc = L.pkv_paged_attention_decode(out.data_ptr(), out.stride(0), out.stride(1), q.data_ptr(), q.stride(0),
                                      q.stride(1), k.data_ptr(), v.data_ptr(), *k.stride()[:3], *k.shape,
                                      tables.data_ptr(), tables.stride(0), tables.shape[1], ctx.data_ptr(), 4, 8, 2500,
                                      128 ** -0.5, native.PKV_FLOAT16, ws.data_ptr(), need, s)
    native.check(rc, "decode")
    torch.cuda.synchronize()
    assert torch.equal(out[1], torch.full_like(out[1], 7.0))
    torch.testing.assert_close(out[[0, 2, 3]].cpu(), ref, atol=2e-3, rtol=2e-3)
    assert int(ws[:256 * 1024].count_nonzero()) == 0


def test_rows_off_16_bytes_are_appended_by_the_append_kernel():
    b = _batch([33, 900, 64], dtype=torch.float16, d=64, bs=16, kv=2, group=2, seed=8)
    plain = _run(b, fused=True)[0]
    wide = torch.zeros(3, 2, 66, dtype=torch.float16)
    odd = dict(b)
    for name in ("k_new", "v_new"):
        w = wide.clone().cuda()
        w[:, :, 2:] = b[name].cuda()
        odd[name] = w[:, :, 2:]
    n, bs = 3, 16
    last = b["ctx"] - 1
    slots = b["tables"][torch.arange(n), last // bs] * bs + last % bs
    kd, vd = b["k"].cuda(), b["v"].cuda()
    out = paged_attention_hip_launch(b["q"].cuda(), kd, vd, b["tables"].cuda(), b["ctx"].cuda(),
                                     torch.ones(n, dtype=torch.long).cuda(), 64 ** -0.5,
                                     append=(odd["k_new"], odd["v_new"], slots.cuda()))
    assert torch.equal(out.cpu(), plain)


#: Around the edges of a block, a wave's 64 tokens and a 256-token partition, up to 5 partitions.
REGISTER_EDGES = [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 271, 320, 321, 511, 512, 513,
                  576, 767, 768, 769, 1000, 1023, 1024, 1025, 1279, 1280]


@pytest.mark.parametrize("kv,group", [(12, 1), (3, 2), (16, 1), (14, 2)])   # the last two past 2048 workgroups
@pytest.mark.parametrize("ctx", [REGISTER_EDGES, REGISTER_EDGES[:15]], ids=["partitions", "one partition"])
@pytest.mark.parametrize("fused", [False, True], ids=["plain", "append"])
def test_fp32_register_kernel(kv, group, ctx, fused):
    """attn_decode.hip: fp32, head_dim 64, groups of 1 and 2."""
    _check(_batch(ctx, dtype=torch.float32, d=64, bs=16, kv=kv, group=group, seed=group), fused=fused)


def test_fp32_register_kernel_appends_rows_off_16_bytes():
    """By the append launch, in front of the same kernel: the same bits."""
    b = _batch(REGISTER_EDGES, dtype=torch.float32, d=64, bs=16, kv=3, group=1)
    out, k, v, slots = _run(b, fused=True)
    kd, vd = b["k"].cuda(), b["v"].cuda()
    odd = [torch.empty(t.numel() + 1, device="cuda")[1:].view(t.shape).copy_(t) for t in (b["k_new"], b["v_new"])]
    assert all(t.data_ptr() % 16 for t in odd)
    got = paged_attention_hip_launch(b["q"].cuda(), kd, vd, b["tables"].cuda(), b["ctx"].cuda(),
                                     torch.ones(len(slots), dtype=torch.long).cuda(), 0.125, append=(*odd, slots.cuda()))
    assert torch.equal(got.cpu(), out)
    assert torch.equal(torch.nan_to_num(kd.cpu()), torch.nan_to_num(k))
    assert torch.equal(torch.nan_to_num(vd.cpu()), torch.nan_to_num(v))


def _captured(b, width, bound):
    """The call captured with `bound` as the longest context, replayed on the real lengths."""
    n = len(b["ctx"])
    tables = torch.zeros(n, width, dtype=torch.long)
    tables[:, :b["tables"].shape[1]] = b["tables"]
    ctx, ones = b["ctx"].cuda(), torch.ones(n, dtype=torch.long)
    attach_host(ctx, torch.full((n,), bound))
    args = (b["q"].cuda(), b["k"].cuda(), b["v"].cuda(), tables.cuda(), ctx, attach_host(ones.cuda(), ones),
            b["q"].shape[2] ** -0.5)
    graph, out, census = capture_step(lambda: paged_attention_hip_launch(*args), torch.device("cuda", 0),
                                      torch.cuda.Stream(), None, "decode")
    out.fill_(float("nan"))
    graph.replay()
    torch.cuda.synchronize()
    return out.cpu(), census


@pytest.mark.parametrize("n,dtype,kv,group,d,bs,lo,hi,bound", [
    (24, torch.float32, 12, 1, 64, 16, 40, 500, 1024), (24, torch.float32, 12, 1, 64, 16, 40, 500, 4096), (8, torch.float32, 6, 2, 64, 16, 40, 300, 1024),
    (32, torch.float32, 4, 4, 64, 16, 40, 500, 1024), (8, torch.float32, 8, 1, 128, 16, 40, 250, 2048),
    (64, torch.float16, 12, 1, 64, 16, 40, 500, 1024), (43, torch.float16, 12, 1, 64, 16, 40, 512, 1024),
    (8, torch.float16, 12, 1, 64, 16, 17, 700, 1024), (64, torch.bfloat16, 8, 4, 128, 16, 30, 250, 1024),
    (8, torch.bfloat16, 8, 4, 128, 16, 30, 520, 4096), (300, torch.bfloat16, 6, 2, 128, 16, 30, 3000, 8192),
    (20, torch.float16, 1, 3, 80, 32, 30, 520, 4096),
    (130, torch.float16, 3, 1, 64, 16, 30, 600, 15000), (130, torch.float16, 3, 1, 64, 32, 30, 11000, 15000)])
def test_a_captured_call_computes_the_eager_one(n, dtype, kv, group, d, bs, lo, hi, bound):
    """Bit for bit, whatever longest context the capture was told: what is cut, and where, comes
    from the lengths."""
    ctx = [lo + i % 7 for i in range(n)]
    for i in range(5):
        ctx[(i * n) // 5] = hi - i
    b = _batch(ctx, dtype=dtype, d=d, bs=bs, kv=kv, group=group, seed=n)
    eager = _run(b, fused=False)[0]
    out, census = _captured(b, -(-bound // bs), bound)
    assert torch.equal(out, eager)
    # One launch, but for the fp32 register kernel's merge at a bound of more than 2048 workgroups.
    registers = dtype == torch.float32 and d == 64 and group <= 2
    assert census == {"kernel": 2 if registers and n * kv * -(-bound // 256) > 2048 else 1}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("far", [16 * 8, 16 * 40 + 5])
def test_the_largest_weight_is_not_rounded(dtype, far):
    """Two keys that nearly cancel, the later one's weight against the first no number of the
    pool dtype: rounded, it would leave nothing of the output. (2e-2 covers the output's own
    rounding and exp2's.)"""
    n, ctx = 12, far + 9
    b = _batch([ctx] * n, dtype=dtype, d=64, bs=16, kv=1, group=1)
    score = torch.tensor([1.0 + 0.34375 * i for i in range(n)]).to(dtype)     # all numbers of both dtypes
    w = score.double().exp()
    b["q"].zero_()[:, :, 0] = 8.0                                              # scores: K's first column
    for i in range(n):
        k, v = torch.zeros(ctx, 64), torch.zeros(ctx, 64)
        k[:, 0] = -100.0
        k[0, 0], k[far, 0] = 0.0, score[i]
        v[0], v[far] = -w[i].to(dtype).float(), 1.0
        pos = torch.arange(ctx)
        at = b["tables"][i, pos // 16], pos % 16
        b["k"][at], b["v"][at] = k.to(dtype)[:, None], v.to(dtype)[:, None]
    want = (w - w.to(dtype).double()) / (1 + w)
    out = _run(b, fused=False)[0].double()
    torch.testing.assert_close(out, want[:, None, None].expand_as(out), rtol=2e-2, atol=1e-6)
