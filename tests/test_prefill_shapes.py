"""The 16-bit prefill kernel on the shapes, groups and block sizes it takes, and its split
contexts, and fp32 prompts of the same shapes (16 rows a workgroup), against oracle.gather
(the reference gather path) at the bars of 2e-2 in 16 bits and 1e-5 in fp32.

Contexts end on, before and behind the edges of a block, an 8-key half, a 64-key tile, a
32-row wave and a 128-row workgroup (query rows are tokens x group heads). Decode batches
of the shapes without a decode kernel run through it too.
"""

from __future__ import annotations

import ctypes
import random

import numpy as np
import pytest
import torch

from inference_server import native
from inference_server.core.attention_hip import _WORKSPACES, attach_host, paged_attention_hip_launch
from oracle.gather import paged_attention_gather as oracle_gather
from oracle.kvops import kv_append

TOL = {torch.float16: 2e-2, torch.bfloat16: 2e-2, torch.float32: 1e-5}
EDGES = [(1, 1), (7, 7), (8, 8), (9, 5), (64, 1), (63, 63), (65, 65), (130, 43), (300, 129), (257, 1)]
DECODE = [(1, 1), (8, 1), (9, 1), (64, 1), (65, 1), (700, 1)]
#: One prompt of a few tiles among contexts long enough to be split.
LONG = [(3000, 1), (1500, 33), (70, 70), (5, 5), (2049, 43), (1025, 2)]


def _batch(lengths, *, dtype, d, bs, kv, group, seed=0):
    g = torch.Generator().manual_seed(seed)
    need = [-(-c // bs) for c, _ in lengths]
    num_blocks = sum(need) + 3
    perm = torch.randperm(num_blocks, generator=g).tolist()
    width = max(need) + 1
    rows = []
    for n in need:
        # Padding past the sequence's blocks is live ids, which a correct kernel never reads.
        rows.append(perm[:n] + torch.randint(0, num_blocks, (width - n,), generator=g).tolist())
        perm = perm[n:]
    t = sum(q for _, q in lengths)
    rand = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    return dict(q=rand(t, kv * group, d), k=rand(num_blocks, bs, kv, d), v=rand(num_blocks, bs, kv, d),
                tables=torch.tensor(rows), ctx=torch.tensor([c for c, _ in lengths]),
                ql=torch.tensor([q for _, q in lengths]), k_new=rand(t, kv, d), v_new=rand(t, kv, d))


def _check(b, *, fused, told=None, scale=None):
    """told: other context lengths for the host copy, which only balances the launch."""
    d, bs = b["q"].shape[2], b["k"].shape[1]
    scale = d ** -0.5 if scale is None else scale
    first = b["ctx"] - b["ql"]
    slots = torch.cat([b["tables"][i, torch.arange(int(f), int(f + n)) // bs] * bs
                       + torch.arange(int(f), int(f + n)) % bs for i, (f, n) in enumerate(zip(first, b["ql"]))])
    k, v = b["k"].cuda(), b["v"].cuda()
    ctx = attach_host(b["ctx"].cuda(), b["ctx"] if told is None else told)
    ql = attach_host(b["ql"].cuda(), b["ql"])
    append = (b["k_new"].cuda(), b["v_new"].cuda(), slots.cuda()) if fused else None
    out = paged_attention_hip_launch(b["q"].cuda(), k, v, b["tables"].cuda(), ctx, ql, scale, append=append)
    torch.cuda.synchronize()
    kr, vr = b["k"], b["v"]
    if fused:
        raw = torch.int32 if kr.dtype == torch.float32 else torch.int16
        bits = lambda t: t.view(raw).numpy()  # noqa: E731
        put = lambda pool, rows: torch.from_numpy(kv_append(bits(pool), bits(rows), slots.numpy()))  # noqa: E731
        kb, vb = put(kr, b["k_new"]), put(vr, b["v_new"])
        assert torch.equal(k.cpu().view(raw), kb) and torch.equal(v.cpu().view(raw), vb)
        kr, vr = kb.view(kr.dtype), vb.view(vr.dtype)
    ref = oracle_gather(b["q"], kr, vr, b["tables"], b["ctx"], b["ql"], scale)
    torch.testing.assert_close(out.cpu(), ref, atol=TOL[out.dtype], rtol=TOL[out.dtype])


def _split_bytes(b):
    t, heads, d = b["q"].shape
    kv = b["k"].shape[2]
    return native.lib().pkv_paged_attention_prefill_workspace_bytes(
        len(b["ctx"]), heads, kv, d, t, b["ctx"].data_ptr(), b["ql"].data_ptr())


@pytest.mark.gpu
@pytest.mark.parametrize("d,bs,kv,group,dtype", [
    (32, 8, 2, 1, torch.float16), (32, 16, 1, 5, torch.bfloat16), (48, 32, 2, 3, torch.float16),
    (64, 8, 2, 3, torch.bfloat16), (64, 64, 1, 4, torch.float16), (64, 16, 2, 6, torch.float16),
    (80, 8, 3, 1, torch.bfloat16), (80, 32, 1, 8, torch.float16), (96, 16, 2, 2, torch.bfloat16),
    (112, 128, 1, 3, torch.float16), (128, 32, 2, 4, torch.bfloat16), (128, 8, 1, 16, torch.float16),
    (128, 16, 1, 71, torch.bfloat16), (128, 16, 2, 3, torch.float16),
    (32, 8, 2, 3, torch.float32), (48, 16, 1, 5, torch.float32), (64, 16, 2, 1, torch.float32),
    (80, 32, 1, 8, torch.float32), (96, 64, 2, 2, torch.float32), (112, 8, 1, 1, torch.float32),
    (128, 16, 1, 71, torch.float32), (128, 32, 2, 4, torch.float32)])
@pytest.mark.parametrize("lengths", [EDGES, DECODE], ids=["prompts", "decode"])
@pytest.mark.parametrize("fused", [False, True], ids=["plain", "append"])
def test_shapes_groups_and_block_sizes(d, bs, kv, group, dtype, lengths, fused):
    _check(_batch(lengths, dtype=dtype, d=d, bs=bs, kv=kv, group=group, seed=d + bs + group), fused=fused)


@pytest.mark.gpu
@pytest.mark.parametrize("d,bs,kv,group,dtype", [
    (64, 16, 2, 1, torch.float16), (128, 16, 2, 4, torch.bfloat16), (48, 8, 2, 3, torch.float16),
    (80, 32, 1, 8, torch.bfloat16), (64, 16, 1, 17, torch.float16), (128, 16, 2, 1, torch.float32),
    (32, 8, 1, 3, torch.float32)])
@pytest.mark.parametrize("scale", [0.0, -0.125])
@pytest.mark.parametrize("lengths", [EDGES, DECODE, LONG], ids=["prompts", "decode", "long"])
def test_scales_that_are_not_positive(d, bs, kv, group, dtype, scale, lengths):
    _check(_batch(lengths, dtype=dtype, d=d, bs=bs, kv=kv, group=group, seed=d + 1), fused=True, scale=scale)


@pytest.mark.gpu
@pytest.mark.parametrize("d,bs,kv,group,dtype", [
    (64, 16, 2, 1, torch.float16), (128, 16, 2, 4, torch.bfloat16), (128, 16, 1, 3, torch.float16),
    (80, 32, 2, 3, torch.bfloat16), (32, 8, 1, 8, torch.float16)])
@pytest.mark.parametrize("fused", [False, True], ids=["plain", "append"])
def test_split_contexts(d, bs, kv, group, dtype, fused):
    b = _batch(LONG, dtype=dtype, d=d, bs=bs, kv=kv, group=group, seed=7 + d)
    assert _split_bytes(b) > 0
    _check(b, fused=fused)
    # A decode batch of long contexts (a decode kernel's where one takes the shape).
    lone = _batch([(c, 1) for c, _ in LONG], dtype=dtype, d=d, bs=bs, kv=kv, group=group, seed=9 + d)
    _check(lone, fused=fused)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,bs,grows", [(torch.float32, 16, 0), (torch.bfloat16, 12, 0), (torch.bfloat16, 16, 1)])
def test_only_batches_that_can_split_grow_the_workspace(dtype, bs, grows):
    b = _batch([(6000, 30)], dtype=dtype, d=64, bs=bs, kv=1, group=4)
    torch.cuda.synchronize()
    _WORKSPACES.reset()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        _check(b, fused=False)
    held = [key for key in _WORKSPACES._bufs if key[1] == stream.cuda_stream]
    assert len(held) == grows


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 65, 200])
def test_fp32_prompts_over_sequence_counts(n):
    """Tiles found across lanes, several sequences a lane, prompts of no token among them."""
    lengths = [(20 + (13 * i) % 90, (7 * i) % 19) for i in range(n)]
    lengths[0], lengths[n // 2], lengths[n - 1] = (1500, 33), (40, 40), (17, 16)
    _check(_batch(lengths, dtype=torch.float32, d=64, bs=16, kv=1, group=3, seed=n), fused=False)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [15, 16, 17, 64, 65, 200, 256, 257])
@pytest.mark.parametrize("split", [False, True], ids=["whole", "split"])
def test_prompts_over_sequence_counts(n, split):
    """Items found within a wave and through LDS, on grids that are not a multiple of 8 items,
    with prompts of no token among them; with and without long contexts to split (257
    sequences never are)."""
    lengths = [(20 + (13 * i) % 90, (7 * i) % 19) for i in range(n)]
    lengths[0], lengths[n // 2], lengths[n - 1] = (1500 if split else 150, 33), (40, 40), (3000 if split else 17, 1)
    b = _batch(lengths, dtype=torch.float16, d=64, bs=16, kv=1, group=3, seed=n)
    assert (_split_bytes(b) > 0) == (split and n <= 256)
    _check(b, fused=True)
    if split:       # the host's lengths only balance the launch: a grid without room for the splits
        told = torch.where(b["ctx"] > 1000, torch.tensor(1100), b["ctx"])
        _check(b, fused=False, told=told)


@pytest.mark.gpu
@pytest.mark.parametrize("told", [[1100] * 6, [3000, 40, 70, 5, 43, 2]], ids=["shorter", "one long"])
def test_split_contexts_longer_than_told_are_attended_whole(told):
    b = _batch(LONG, dtype=torch.bfloat16, d=128, bs=16, kv=2, group=4, seed=11)
    told = torch.tensor(told)
    heads, kv = 8, 2
    assert native.lib().pkv_paged_attention_prefill_workspace_bytes(
        len(told), heads, kv, 128, b["q"].shape[0], told.data_ptr(), b["ql"].data_ptr()) > 0
    _check(b, fused=False, told=told)


def test_split_workspace_is_host_arithmetic():
    size = native.lib().pkv_paged_attention_prefill_workspace_bytes
    arr = lambda v: (ctypes.c_int64 * len(v))(*v)  # noqa: E731

    def need(ctx, ql, heads=32, kv=8, d=128):
        return size(len(ctx), heads, kv, d, sum(ql), arr(ctx), arr(ql))

    assert need([8192], [16]) > 256 * 1024                      # one long context: split
    assert need([1024], [16]) == 0                              # no context past the shortest split one
    assert need([4096] * 16, [512] * 16) == 0                   # the GPU is full without
    assert need([8192] * 257, [1] * 257) == 0                   # more sequences than are ordered
    assert need([8192], [16], heads=3, kv=2) == 0               # not a group
    assert size(1, 32, 8, 128, 16, None, None) == 0
    # Partials stay bounded whatever the batch.
    for n in (1, 3, 12, 100):
        for ctx in (2000, 8192, 131072):
            for q in (1, 40, 300):
                assert need([ctx] * n, [q] * n) <= (130 << 20) + 8 * n * q * 32 + (1 << 20)


@pytest.mark.gpu
@pytest.mark.parametrize("d,bs,dtype", [(128, 16, torch.bfloat16), (80, 32, torch.float16), (64, 16, torch.float32)])
@pytest.mark.parametrize("lengths", [EDGES, DECODE], ids=["prompts", "decode"])
def test_slots_of_a_block_in_reverse_order(d, bs, dtype, lengths):
    """A pool whose slot stride is negative (C ABI only: torch has no such strides)."""
    b = _batch(lengths, dtype=dtype, d=d, bs=bs, kv=2, group=2, seed=d)
    k, v = b["k"].flip(1).contiguous().cuda(), b["v"].flip(1).contiguous().cuda()
    back = (bs - 1) * k.stride(1) * k.element_size()
    q, tables, ctx = b["q"].cuda(), b["tables"].cuda(), b["ctx"].cuda()
    out = torch.full_like(q, float("nan"))
    code, L, s = native.dtype_code(dtype), native.lib(), torch.cuda.current_stream().cuda_stream
    args = (out.data_ptr(), out.stride(0), out.stride(1), q.data_ptr(), q.stride(0), q.stride(1),
            k.data_ptr() + back, v.data_ptr() + back, k.stride(0), -k.stride(1), k.stride(2), *k.shape,
            tables.data_ptr(), tables.stride(0), tables.shape[1], ctx.data_ptr())
    n, heads = len(lengths), q.shape[1]
    if lengths is DECODE:
        need = L.pkv_paged_attention_decode_workspace_bytes(n, heads, 2, d, 700)
        ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
        rc = L.pkv_paged_attention_decode(*args, n, heads, 700, d ** -0.5, code, ws.data_ptr(), need, s)
    else:
        qsl = torch.tensor([0, *torch.cumsum(b["ql"], 0).tolist()]).cuda()
        rc = L.pkv_paged_attention_prefill(*args, qsl.data_ptr(), n, heads, q.shape[0], int(b["ql"].max()), d ** -0.5,
                                           code, s)
    native.check(rc, "attention")
    torch.cuda.synchronize()
    ref = oracle_gather(b["q"], b["k"], b["v"], b["tables"], b["ctx"], b["ql"], d ** -0.5)
    torch.testing.assert_close(out.cpu(), ref, atol=TOL[dtype], rtol=TOL[dtype])


def test_shapes_that_cannot_be_split_take_no_workspace():
    can = native.lib().pkv_paged_attention_prefill_can_split
    fp16, bf16, fp32 = native.PKV_FLOAT16, native.PKV_BFLOAT16, native.PKV_FLOAT32
    assert all(can(bs, d, t) for bs in (8, 16, 128) for d in (32, 48, 128) for t in (fp16, bf16))
    assert not any(can(16, d, fp32) for d in (32, 64, 128))
    assert not any(can(bs, 64, fp16) for bs in (0, 1, 4, 6, 24, 48)) and not any(can(16, d, bf16) for d in (8, 40, 144))


def _planned_bytes(ctx, ql, heads, kv, d):
    """The workspace of the cheapest run length in the launch model of csrc/attn_prefill.hip,
    computed sequence by sequence in whole numbers."""
    up = lambda a, b: -(-a // b)  # noqa: E731
    group, slots = heads // kv, 512 if d >= 112 else 768 if d >= 80 else 1024
    live = [(up(c, 64), up(q * group, 128) * kv, q * heads) for c, q in zip(ctx, ql) if c > 0 and q > 0]
    f = np.float32

    def us(wgs, longest, work):
        tile = f(1.1) + (f(1.9) - f(1.1)) * (f(wgs) / f(slots) if wgs < slots else f(1))
        one = f(longest) * tile + f(6)
        return one if wgs <= slots else max(one, (f(work) * tile + f(wgs) * f(6)) / f(slots) + f(0.5) * one)

    wgs, work, longest = sum(w for _, w, _ in live), sum(t * w for t, w, _ in live), max(t for t, _, _ in live)
    if len(ctx) > 256 or wgs >= 2 * slots or longest * 64 <= 1024:
        return 0
    rows, splits, best = sum(ql) * heads, 1, f(0.85) * us(wgs, longest, work)
    for run in (4, 5, 6, 8, 10, 12, 14, 17, 20, 24, 28, 34, 40, 48, 56, 68, 80, 96, 112, 136, 160, 192):
        if run >= longest:
            break
        n = up(longest, run)
        if 256 * 1024 + 3 * 256 + rows * 4 + rows * n * (d + 2) * 4 > 128 << 20:
            continue
        s = [up(t, run) for t, _, _ in live]
        parts = sum(r * m for (_, _, r), m in zip(live, s) if m > 1)
        cost = us(sum(w * m for (_, w, _), m in zip(live, s)), max(up(t, m) for (t, _, _), m in zip(live, s)), work)
        cost = cost + f(4) + f(parts * (d + 2) * 4) / f(4.5e6)
        if cost < best:
            best, splits = cost, n
    r256 = lambda b: up(b, 256) * 256  # noqa: E731
    return 0 if splits == 1 else 256 * 1024 + r256(rows * 4) + r256(rows * splits * 8) + r256(rows * splits * d * 4)


def test_split_plan_is_the_cheapest_run_length():
    size = native.lib().pkv_paged_attention_prefill_workspace_bytes
    rng, split = random.Random(7), 0
    for _ in range(600):
        n, kv, d = rng.choice([1, 2, 3, 5, 16, 64, 101, 256]), rng.choice([1, 2, 4, 8]), rng.choice([32, 80, 128])
        heads, q, hi = kv * rng.choice([1, 3, 4, 17]), rng.choice([1, 4, 40, 300]), rng.choice([1500, 8192, 131072])
        ql = [rng.randint(n > 1, q) for _ in range(n)]
        ql[0] = max(ql[0], 1)
        ctx = [max(m, rng.randint(1, hi)) for m in ql]
        arr = lambda v: (ctypes.c_int64 * n)(*v)  # noqa: E731
        need = size(n, heads, kv, d, sum(ql), arr(ctx), arr(ql))
        assert need == _planned_bytes(ctx, ql, heads, kv, d), (n, heads, kv, d, ql, ctx)
        assert need <= 128 << 20
        split += need > 0
    assert split > 200
