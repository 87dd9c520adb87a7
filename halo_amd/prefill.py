"""Chunked causal prefill attention on MFMA (bf16, fp16, fp32).

``prefill_attention(q, chunks)`` attends a block of query rows to a list of
KV chunks (prior context chunks plus the query block's own K/V, the latter
causal) and returns the output, optionally with the log-sum-exp, in one
call of ``halo_prefill_attn_split``: one launch, or a few key splits and
their merge where the query rows alone do not fill the GPU.  fp32 queries
(the reference computes every T_q in fp32, halo/kv_cache_chunked.py:241-276)
take the fp32 matrix instructions.  fp32 calls whose chunks that kernel does
not read (``_f32_direct``) run on the decode kernel: the query rows of each
batch row are the batch of one ``halo_decode_attn`` launch whose chunk
descriptors repeat the same K/V for every such row (batch stride 0), with the
causal position of row i at q_start + i; it reads K/V once per query row.

Reference: the chunked prefill path of HALOCacheChunked.compute_attention
(halo/kv_cache_chunked.py:864-964), which runs _chunk_attention per chunk and
folds the partials with _lse_merge (:194-276); the causal rule is
chunk_start + t <= q_start + i (halo/triton_chunked.py:114-119) and the
default query offset is T_total - T_q (halo/kv_cache_chunked.py:839-840).
"""
from __future__ import annotations

import math
from typing import Optional, Sequence

import numpy as np
import torch

from . import _native as nat
from .decode import ChunkRef, _to_device, descs_to_device, pack_descs


def prefill_attention(q: torch.Tensor, chunks: Sequence[ChunkRef], *, scale: Optional[float] = None,
                      q_start=None, out_dtype: Optional[torch.dtype] = None, return_lse: bool = False,
                      stream=None):
    """q (B, H, T_q, D) bf16, fp16 or fp32; chunks (B, H_kv, T_c, D) of the same dtype.
    Returns out (B, H, T_q, D) in ``out_dtype`` (default q.dtype) and, with
    ``return_lse``, lse (B, H, T_q) fp32.  With ``stream``, the inputs are
    read and the results written there."""
    L = nat.lib()
    if q.dim() != 4:
        raise AssertionError(f"q must be (B, H, T_q, D), got {tuple(q.shape)}")
    B, H, T_q, D = q.shape
    if not chunks:
        raise AssertionError("no chunks to attend")
    if q.dtype == torch.float32 and not _f32_direct(q, chunks):
        return _prefill_fp32_rows(q, chunks, scale=scale, q_start=q_start, out_dtype=out_dtype,
                                  return_lse=return_lse, stream=stream)
    if q.dtype not in (torch.bfloat16, torch.float16, torch.float32):
        raise AssertionError(f"prefill runs on bf16, fp16 or fp32; got {q.dtype}")
    H_kv = chunks[0].k.shape[-3]
    if H % H_kv:
        raise AssertionError(f"head count mismatch: q has {H}, kv has {H_kv}")
    scale = 1.0 / math.sqrt(D) if scale is None else float(scale)
    if q_start is None:
        q_start = sum([c.T for c in chunks]) - T_q
    if q.dtype == torch.float32 and torch.is_tensor(q_start) and q_start.numel() not in (1, B):
        raise AssertionError(f"q_start must have B={B} entries")
    descs, keep = pack_descs(chunks, B=B, H_kv=H_kv, D=D, dtype=q.dtype)
    # A copy of q, the uploads and the launch share one stream (the caller's,
    # or the current one), so the kernel sees them; copy and tables are freed
    # into torch's stream-ordered caching allocator on that stream.  q_start gets
    # there without a blocking copy (a pageable host-to-device copy would
    # hold the host until the stream drains); a plain number goes behind the
    # descriptors in their copy (a fill of its own was 4 us of host and 2-4 us
    # of GPU time in front of every call).  The caller owns the K/V.
    with torch.cuda.stream(stream) if stream is not None else _nullctx():
        q = _aligned_q(q)
        qs_b, qs_h, qs_t = (st if n > 1 else 0 for st, n in zip(q.stride()[:3], q.shape)) if q.dtype == torch.float32 \
            else q.stride()[:3]
        if torch.is_tensor(q_start):
            if q_start.device.type != "cuda":
                q_start = _to_device(q_start.to(torch.int64).reshape(-1).expand(B).numpy(), q.device)
            if q.dtype == torch.float32 and q_start.numel() == 1:
                q_start = q_start.reshape(1).expand(B)
            q_start = q_start.to(device=q.device, dtype=torch.int64).reshape(B).contiguous()
            d_descs = descs_to_device(descs, q.device)
            starts = q_start.data_ptr()
        else:
            table = np.empty(descs.nbytes + 8 * B, np.uint8)
            table[:descs.nbytes] = descs.view(np.uint8)
            table[descs.nbytes:].view(np.int64)[:] = int(q_start)
            d_descs = _to_device(table, q.device)
            starts = d_descs.data_ptr() + descs.nbytes
        out = torch.empty((B, H, T_q, D), device=q.device, dtype=out_dtype or q.dtype)
        lse = torch.empty((B, H, T_q), device=q.device, dtype=torch.float32) if return_lse else None
        dt = nat.dtype_code(q.dtype)
        n_split = L.halo_prefill_splits(dt, B, H, H_kv, T_q, D, *_longest_walk(chunks))
        ws_bytes = L.halo_prefill_workspace_size(dt, B, H, H_kv, T_q, D, n_split)
        try:
            ws = torch.empty(ws_bytes, device=q.device, dtype=torch.uint8) if ws_bytes else None
        except torch.OutOfMemoryError:  # the unsplit walk needs none
            n_split, ws_bytes, ws = 1, 0, None
        nat.check(L.halo_prefill_attn_split(
            q.data_ptr(), qs_b, qs_h, qs_t, dt, B, H, H_kv, T_q, D,
            starts, d_descs.data_ptr(), len(chunks), scale,
            out.data_ptr(), out.stride(0), out.stride(1), out.stride(2), nat.dtype_code(out.dtype),
            nat.ptr(lse), n_split, nat.ptr(ws), ws_bytes, nat.stream_ptr(stream)), "halo_prefill_attn_split")
    del keep
    return (out, lse) if return_lse else out


def _longest_walk(chunks: Sequence[ChunkRef]) -> tuple[int, int]:
    """(keys, keys in causal chunks) of the batch row that attends most keys."""
    keys = causal = 0
    own: dict = {}
    for c in chunks:
        n = c.T
        if c.batch < 0:
            keys += n
            if c.causal:
                causal += n
        else:
            k, d = own.get(c.batch, (0, 0))
            own[c.batch] = (k + n, d + n if c.causal else d)
    k, d = max(own.values(), default=(0, 0))
    return keys + k, causal + d


def _aligned_q(q: torch.Tensor) -> torch.Tensor:
    if q.dtype != torch.float32:
        return q.contiguous() if q.stride(-1) != 1 or (q.stride(-2) * 2) % 16 or q.data_ptr() % 16 else q
    odd = q.stride(-1) != 1 or q.data_ptr() % 16 or any(n > 1 and st % 4 for st, n in zip(q.stride()[:3], q.shape))
    return q.clone(memory_format=torch.contiguous_format) if odd else q


def _f32_direct(q: torch.Tensor, chunks: Sequence[ChunkRef]) -> bool:
    """Whether the fp32 MFMA kernel takes the call: head dim 64 or 128 and
    chunks of the batch whose rows and heads are 16-byte aligned and do not
    overlap, with row strides that a tile's buffer offsets can hold.  The
    decode kernel's row-by-row form keeps the others, and their errors."""
    B, H, T_q, D = q.shape
    if B == 0 or T_q == 0 or D not in (64, 128) or not q.is_cuda:
        return False
    for c in chunks:
        for t in (getattr(c, "k", None), getattr(c, "v", None)):
            if t is None or t.dim() != 4 or t.shape[0] != B or t.shape[-1] != D or t.dtype != torch.float32:
                return False
            if getattr(c, "batch", 0) >= 0 or t.stride(-1) != 1 or t.data_ptr() % 16:
                return False
            sb, sh, st = t.stride()[:3]
            if (t.shape[0] > 1 and sb % 4) or (t.shape[1] > 1 and sh % 4) or st % 4 or not D <= st < 1 << 22:
                return False
    return True


def _prefill_fp32_rows(q: torch.Tensor, chunks: Sequence[ChunkRef], *, scale, q_start, out_dtype,
                       return_lse: bool, stream):
    """fp32 prefill as one decode launch per batch row: pseudo-batch row i is
    query row i, every chunk is read through a batch stride of 0, and the
    causal cut of row i is q_start + i."""
    from .decode import build_plan, launch
    B, H, T_q, D = q.shape
    H_kv = chunks[0].k.shape[-3]
    if H % H_kv:
        raise AssertionError(f"head count mismatch: q has {H}, kv has {H_kv}")
    scale = 1.0 / math.sqrt(D) if scale is None else float(scale)
    if q_start is None:
        q_start = sum(c.T for c in chunks) - T_q
    if torch.is_tensor(q_start):
        starts = [int(x) for x in q_start.reshape(-1).tolist()]
        if len(starts) == 1:
            starts = starts * B
    else:
        starts = [int(q_start)] * B
    if len(starts) != B:
        raise AssertionError(f"q_start must have B={B} entries")
    with torch.cuda.stream(stream) if stream is not None else _nullctx():
        out = torch.empty((B, H, T_q, D), device=q.device, dtype=out_dtype or q.dtype)
        lse = torch.empty((B, H, T_q), device=q.device, dtype=torch.float32) if return_lse else None
        for b in range(B):
            rows = []
            for c in chunks:
                if c.k.dtype != torch.float32 or c.v.dtype != torch.float32:
                    raise AssertionError(f"fp32 query needs fp32 chunks, got {c.k.dtype}/{c.v.dtype}")
                kb, vb = c.k[b:b + 1], c.v[b:b + 1]
                rows.append(ChunkRef(kb.expand(T_q, *kb.shape[1:]), vb.expand(T_q, *vb.shape[1:]),
                                     int(c.chunk_start), bool(c.causal)))
            q_pos_host = [starts[b] + i for i in range(T_q)]
            plan = build_plan(B=T_q, H=H, H_kv=H_kv, D=D, dtype=torch.float32, chunks=rows, device=q.device,
                              q_pos_host=q_pos_host)
            q_pos = torch.arange(starts[b], starts[b] + T_q, dtype=torch.int64).to(q.device, non_blocking=True)
            o_b = torch.empty((T_q, H, D), device=q.device, dtype=out.dtype)
            l_b = torch.empty((T_q, H), device=q.device, dtype=torch.float32) if return_lse else None
            launch(plan, q[b].transpose(0, 1), scale=scale, q_pos=q_pos, out=o_b, lse=l_b)
            out[b].copy_(o_b.transpose(0, 1))
            if return_lse:
                lse[b].copy_(l_b.transpose(0, 1))
    return (out, lse) if return_lse else out


class _nullctx:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False
