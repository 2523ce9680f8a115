"""ATTENTION=hip: paged attention on libpagedkv's CDNA4 kernels.

Same signature, contract checks and exception texts as the gather path
(core/attention.py). Differences are in where the checks read the lengths and in
what runs afterwards:

* Lengths. The reference's `_check` reads context_lens/query_lens back from the
  device with three to four host syncs per call (reference core/attention.py:212-218).
  Here a caller that already holds the lengths on the host (the paged executor
  builds them from Python lists) attaches them with `attach_host`; the checks then
  run with no device round trip. Without an attached copy one combined D2H copy is
  made, and CPU tensors are used as they are.
* Kernels. An all-decode batch (every query_len == 1) goes to
  pkv_paged_attention_decode (split-KV, GQA-shared K/V reads); any other batch goes
  to pkv_paged_attention_prefill. Both accept the strided query view the executor
  hands over (`query[0].transpose(0, 1)`, reference core/paged_executor.py:146)
  without a copy.
* No fallback. Without the library or a ROCm device this raises
  NotImplementedError, like the reference's Triton launcher
  (core/attention_triton.py:254-264).
"""

from __future__ import annotations

import threading

import numpy as np
import torch

from inference_server import native
from inference_server.core.attention import check_contract

_HOST_ATTR = "_pkv_host"


def attach_host(device_tensor: torch.Tensor, host_tensor: torch.Tensor) -> torch.Tensor:
    """Record a host (CPU) copy of `device_tensor`'s values for host-side checks.
    The caller guarantees the two hold the same values. Returns device_tensor."""
    setattr(device_tensor, _HOST_ATTR, host_tensor)
    return device_tensor


_QSL_ATTR = "_pkv_qsl"


def attach_query_start(query_lens: torch.Tensor, query_start: torch.Tensor) -> torch.Tensor:
    """Record the device query_start_loc [B+1] (0, then the running sum of query_lens)
    that a prefill launch should use instead of building one from the host lengths
    (a caller that keeps its metadata in persistent device buffers, such as a captured
    graph, supplies it). The caller guarantees the values match. Returns query_lens."""
    setattr(query_lens, _QSL_ATTR, query_start)
    return query_lens


def host_copy(t: torch.Tensor) -> torch.Tensor | None:
    if t.device.type == "cpu":
        return t
    return getattr(t, _HOST_ATTR, None)


def _host_lengths(context_lens: torch.Tensor, query_lens: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    hc, hq = host_copy(context_lens), host_copy(query_lens)
    if hc is None or hq is None:
        both = torch.stack([context_lens.reshape(-1).long(), query_lens.reshape(-1).long()]).cpu()
        hc, hq = both[0], both[1]
    return hc.long().contiguous(), hq.long().contiguous()


#: The merge counters at the front of a workspace, what must read zero (include/pagedkv.h).
_COUNTER_BYTES = 256 * 1024


class _Workspaces:
    """One attention workspace per (device, stream), grown on demand and reused across
    calls (split-KV decode and split prefill; a stream runs one call at a time). It is
    zero-filled when allocated: the decode merge counters at its front must read zero when
    a call starts, and every completed call leaves them zero again (the partials behind
    them need no initialisation). A different stream gets its own buffer. Sizes are powers
    of two and a buffer that had to grow is kept, not freed: a graph captured on that
    stream earlier replays into it (the kept ones add up to less than the one in use).
    A capture that finds none large enough gets one of its own, shared by its later calls
    and cleared once, at its first call, by every replay (one fill node, not one a layer).
    After a call that did not complete (a launch error, a reset device), `reset()` drops the
    buffers so the next call gets a zero-filled one."""

    def __init__(self) -> None:
        self._lock = threading.Lock()
        self._bufs: dict[tuple[int, int], torch.Tensor] = {}
        self._kept: list[torch.Tensor] = []
        # (capture id, buffer) of the capture under way on a stream.
        self._captured: dict[tuple[int, int], tuple[int, torch.Tensor]] = {}

    def partials(self, device: torch.device, stream: int, nbytes: int) -> torch.Tensor:
        idx = device.index if device.index is not None else torch.cuda.current_device()
        key = (idx, stream)
        with self._lock:
            buf = self._bufs.get(key)
            if buf is None or buf.numel() < nbytes:
                if torch.cuda.is_current_stream_capturing():
                    capture = native.stream_capture_id(stream)
                    held = self._captured.get(key)
                    if held is None or held[0] != capture or held[1].numel() < nbytes:
                        own = torch.empty(max(nbytes, 1 << 16), dtype=torch.uint8, device=device)
                        own[:_COUNTER_BYTES].zero_()
                        held = self._captured[key] = (capture, own)
                    return held[1]
                self._captured.pop(key, None)
                size = 1 << (max(nbytes, 1 << 16) - 1).bit_length()
                if buf is not None:
                    self._kept.append(buf)
                buf = torch.zeros(size, dtype=torch.uint8, device=device)
                self._bufs[key] = buf
            return buf

    def reset(self) -> None:
        """Forget every buffer (the next call on each stream allocates a zeroed one)."""
        with self._lock:
            self._bufs.clear()
            self._kept.clear()
            self._captured.clear()


_WORKSPACES = _Workspaces()


def _on_device(t: torch.Tensor, dev: torch.device) -> torch.Tensor:
    """t as int64 on dev: itself when it is (the no-op `.to` costs a microsecond)."""
    return t if t.dtype is torch.long and t.device == dev else t.to(device=dev, dtype=torch.long)


_META_ATTR = "_pkv_step_meta"


def _batch_facts(context_lens: torch.Tensor, query_lens: torch.Tensor, block_size: int, width: int) -> dict:
    """Host-side facts about one batch's lengths: the contract checks' inputs, the
    decode/prefill choice, the maxima that size the grids. The paged executor hands
    the same length tensors, with host copies attached, to every layer of a step, so
    for attached tensors the facts are kept on context_lens, keyed by the values of both
    host copies (new values, attached or written in place, make new facts). Tensors
    without attached copies are read afresh on every call."""
    hc_att, hq_att = host_copy(context_lens), host_copy(query_lens)
    key = None
    if hc_att is not None and hq_att is not None and context_lens.device.type != "cpu" and not (
            hc_att.is_cuda or hq_att.is_cuda):
        hc, hq = hc_att.numpy(), hq_att.numpy()
        key = (hc.tobytes(), hq.tobytes(), hc.dtype, hq.dtype, block_size, width)
        hit = getattr(context_lens, _META_ATTR, None)
        if hit is not None and hit[0] == key:
            return hit[1]
    if key is None:
        hc, hq = (t.numpy() for t in _host_lengths(context_lens, query_lens))
    # Copies: facts are kept past this call, and the caller's tensors may be written to. In
    # numpy: the same operations on small tensors took 58-73 us of a first call (16 so).
    hctx, hql = np.array(hc, dtype=np.int64), np.array(hq, dtype=np.int64)
    longest = int(hctx.max()) if hctx.size else 0
    facts = {
        "hctx": torch.from_numpy(hctx),
        "hql": torch.from_numpy(hql),
        "total": int(hql.sum()),
        "q_gt_c": bool((hql > hctx).any()),
        "too_few_blocks": longest > width * block_size,
        "all_decode": bool((hql == 1).all()),
        "max_ctx": longest,
        "max_q": int(hql.max()) if hql.size else 0,
        "split_ws": {},  # split prefill's workspace bytes by shape, planned on first use
        "qsl": {},  # device query_start_loc by (device, stream), built on first prefill use
    }
    if key is not None:
        setattr(context_lens, _META_ATTR, (key, facts))
    return facts


_CAPTURED_ATTR = "_pkv_captured_qsl"


def _query_start(facts: dict, context_lens: torch.Tensor, dev: torch.device, stream: int) -> torch.Tensor:
    """Device query_start_loc of a batch, uploaded once per step and stream. The upload
    leaves from pinned memory: a pageable one waits for everything queued on the stream,
    which cost a step one such wait per layer (3 GPT-2 prompts, 31 us a call of which the
    kernel is 12)."""
    capturing = torch.cuda.is_current_stream_capturing()
    if capturing:
        # A capture takes the one that a call before it uploaded (on any stream: whoever
        # captures has joined the warm-up). It then lives as long as context_lens, which the
        # graph reads too, not only until the facts change. Without one the upload below is
        # refused by the runtime.
        for (where, _), qsl in facts["qsl"].items():
            if where == dev:
                kept = getattr(context_lens, _CAPTURED_ATTR, ())
                if not any(t is qsl for t in kept):
                    setattr(context_lens, _CAPTURED_ATTR, (*kept, qsl))
                return qsl
    qsl = facts["qsl"].get((dev, stream))
    if qsl is None:
        hql = facts["hql"]
        host = torch.zeros(hql.numel() + 1, dtype=torch.long, pin_memory=not capturing)
        torch.cumsum(hql, 0, out=host[1:])
        qsl = host.to(dev, non_blocking=not capturing)
        if not capturing:
            facts["qsl"][(dev, stream)] = qsl
    return qsl


def paged_attention_hip_launch(
    query: torch.Tensor,
    k_pool: torch.Tensor,
    v_pool: torch.Tensor,
    block_tables: torch.Tensor,
    context_lens: torch.Tensor,
    query_lens: torch.Tensor,
    scale: float,
    append: tuple[torch.Tensor, torch.Tensor, torch.Tensor] | None = None,
) -> torch.Tensor:
    """The hip backend of `paged_attention`. With `append` = (k_new, v_new, slots) — the
    batch's new rows [T, Hkv, D] (one per query token) and their flat slots, already
    range-checked — the rows are written into the pool inside the attention call: on a
    decode batch `pkv_paged_attention_decode_append` (the decode kernel stores each row
    from the wave that reads it), on any other batch `pkv_paged_attention_prefill_append`
    (the MFMA kernel stages new positions from the rows themselves and each workgroup
    writes its own tokens' rows), so the step has no separate append launch."""
    native.require_gpu(query, "paged_attention")
    q_shape, p_shape, t_shape = query.shape, k_pool.shape, block_tables.shape
    bs = p_shape[1] if len(p_shape) == 4 else 1
    width = t_shape[1] if len(t_shape) == 2 else 0
    facts: dict | None = None

    def values():
        nonlocal facts
        facts = _batch_facts(context_lens, query_lens, bs, width)
        return facts["total"], facts["q_gt_c"], facts["too_few_blocks"]

    check_contract(len(q_shape), q_shape, len(p_shape), p_shape, t_shape, context_lens.shape, query_lens.shape, values)
    if p_shape != v_pool.shape:
        raise ValueError(f"k_pool {tuple(p_shape)} and v_pool {tuple(v_pool.shape)} differ")
    dev, dtype = query.device, query.dtype
    for name, t in (("k_pool", k_pool), ("v_pool", v_pool)):
        if t.device != dev:
            raise ValueError(f"{name} is on {t.device}, query is on {dev}")
        if t.dtype != dtype:
            raise ValueError(f"{name} dtype {t.dtype} differs from query dtype {dtype}")
    n_tok, n_heads, head_dim = q_shape
    n_blocks, block_size, n_kv, pool_dim = p_shape
    if pool_dim != head_dim:
        raise ValueError(f"query head_dim {head_dim} != pool head_dim {pool_dim}")
    if n_heads % n_kv:
        raise ValueError(f"{n_heads} query heads not divisible by {n_kv} kv heads")
    dt = native.dtype_code(dtype)

    out = torch.empty(q_shape, dtype=dtype, device=dev)
    n_seqs = t_shape[0]
    if n_tok == 0 or n_seqs == 0:
        return out

    if query.stride(2) != 1:
        query = query.contiguous()
    k_st = k_pool.stride()
    if k_st[3] != 1 or v_pool.stride() != k_st:
        if append is not None:
            # A fused append writes the new rows into the pool in place; a contiguous
            # copy of the pool would take the rows and be thrown away.
            raise ValueError("a fused append needs k_pool and v_pool with unit head_dim stride and equal strides; "
                             f"got {tuple(k_st)} and {tuple(v_pool.stride())}")
        k_pool, v_pool = k_pool.contiguous(), v_pool.contiguous()
        k_st = k_pool.stride()
    tables = _on_device(block_tables, dev)
    t_st = tables.stride()
    if t_st[1] != 1:
        tables = tables.contiguous()
        t_st = tables.stride()
    ctx_dev = _on_device(context_lens, dev).contiguous()

    L = native.lib()
    stream = native.stream_handle(dev)
    o_st, q_st = out.stride(), query.stride()
    rows = (out.data_ptr(), o_st[0], o_st[1], query.data_ptr(), q_st[0], q_st[1])
    common_pool = (k_pool.data_ptr(), v_pool.data_ptr(), k_st[0], k_st[1], k_st[2],
                   n_blocks, block_size, n_kv, head_dim,
                   tables.data_ptr(), t_st[0], t_shape[1])
    if append is not None:
        k_new, v_new, slots = append
        if k_new.shape != (n_tok, n_kv, head_dim) or v_new.shape != k_new.shape:
            raise ValueError(f"a fused append needs one new row [{n_kv}, {head_dim}] per query token; "
                             f"got {tuple(k_new.shape)} and {tuple(v_new.shape)} for {n_tok} tokens")
        if k_new.stride(2) != 1 or v_new.stride() != k_new.stride():
            k_new, v_new = k_new.contiguous(), v_new.contiguous()
        slots = _on_device(slots, dev)
    if facts["all_decode"] and append is not None:
        max_ctx = facts["max_ctx"]
        ws_bytes = L.pkv_paged_attention_decode_workspace_bytes(n_seqs, n_heads, n_kv, head_dim, max_ctx)
        ws = _WORKSPACES.partials(dev, stream, ws_bytes)
        rc = L.pkv_paged_attention_decode_append(
            *rows,
            *common_pool[:9],
            k_new.data_ptr(), v_new.data_ptr(), k_new.stride(0), k_new.stride(1), slots.data_ptr(),
            *common_pool[9:],
            ctx_dev.data_ptr(),
            n_seqs, n_heads, max_ctx,
            float(scale), dt,
            ws.data_ptr(), ws.numel(),
            stream,
        )
        native.check(rc, "pkv_paged_attention_decode_append")
        return out
    if facts["all_decode"]:
        max_ctx = facts["max_ctx"]
        ws_bytes = L.pkv_paged_attention_decode_workspace_bytes(n_seqs, n_heads, n_kv, head_dim, max_ctx)
        ws = _WORKSPACES.partials(dev, stream, ws_bytes)
        rc = L.pkv_paged_attention_decode(
            *rows,
            *common_pool,
            ctx_dev.data_ptr(),
            n_seqs, n_heads, max_ctx,
            float(scale), dt,
            ws.data_ptr(), ws.numel(),
            stream,
        )
        native.check(rc, "pkv_paged_attention_decode")
        return out

    qsl = getattr(query_lens, _QSL_ATTR, None)
    if qsl is None:
        qsl = _query_start(facts, context_lens, dev, stream)
    # Workspace for split contexts (0 bytes: a batch that is not split), planned by a step's
    # first layer.
    lens = (facts["hctx"].data_ptr(), facts["hql"].data_ptr())
    shape = (n_heads, n_kv, head_dim, block_size, dt)
    ws_bytes = facts["split_ws"].get(shape)
    if ws_bytes is None:
        ws_bytes = 0
        if L.pkv_paged_attention_prefill_can_split(block_size, head_dim, dt):
            ws_bytes = L.pkv_paged_attention_prefill_workspace_bytes(n_seqs, n_heads, n_kv, head_dim, n_tok, *lens)
        facts["split_ws"][shape] = ws_bytes
    ws_ptr, ws_size = None, 0
    if ws_bytes:
        ws = _WORKSPACES.partials(dev, stream, ws_bytes)
        ws_ptr, ws_size = ws.data_ptr(), ws.numel()
    new = (None, None, 0, 0, None) if append is None else (
        k_new.data_ptr(), v_new.data_ptr(), k_new.stride(0), k_new.stride(1), slots.data_ptr())
    rc = L.pkv_paged_attention_prefill_split(
        *rows,
        *common_pool[:9],
        *new,
        *common_pool[9:],
        ctx_dev.data_ptr(), qsl.data_ptr(),
        n_seqs, n_heads, n_tok, facts["max_q"], *lens,
        float(scale), dt,
        ws_ptr, ws_size,
        stream,
    )
    native.check(rc, "pkv_paged_attention_prefill")
    return out
