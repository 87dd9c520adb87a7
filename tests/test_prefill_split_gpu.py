"""The split walk of the chunked prefill: n_split partial passes and their
merge against the float64 closed form, at the edges of the split ranges."""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import attention as A
from oracle.inputs import round_to

pytestmark = pytest.mark.gpu

DT = {"bfloat16": torch.bfloat16, "float16": torch.float16}


def _split(q, chunks, n_split, *, q_start, out_dtype=torch.float32):
    from halo_amd import _native as nat
    from halo_amd.decode import descs_to_device, pack_descs
    L = nat.lib()
    B, H, T_q, D = q.shape
    H_kv = chunks[0].k.shape[-3]
    descs, keep = pack_descs(chunks, B=B, H_kv=H_kv, D=D, dtype=q.dtype)
    dd = descs_to_device(descs, q.device)
    qs = torch.full((B,), q_start, device=q.device, dtype=torch.int64)
    out = torch.full((B, H, T_q, D), float("nan"), device=q.device, dtype=out_dtype)
    lse = torch.full((B, H, T_q), float("nan"), device=q.device)
    nb = L.halo_prefill_workspace_size(B, H, H_kv, T_q, D, n_split)
    ws = torch.full((max(nb, 16),), 0xFF, device=q.device, dtype=torch.uint8)
    nat.check(L.halo_prefill_attn_split(
        q.data_ptr(), *q.stride()[:3], nat.dtype_code(q.dtype), B, H, H_kv, T_q, D, qs.data_ptr(), dd.data_ptr(),
        len(chunks), 1 / math.sqrt(D), out.data_ptr(), *out.stride()[:3], nat.dtype_code(out.dtype), lse.data_ptr(),
        n_split, ws.data_ptr(), nb, nat.stream_ptr()), "halo_prefill_attn_split")
    torch.cuda.synchronize()
    return out.cpu().numpy(), lse.cpu().numpy()


@pytest.mark.parametrize("dtype,B,H,H_kv,D,T_prior,T_q,chunk", [
    ("bfloat16", 1, 8, 2, 128, 384, 130, 128),   # a second, nearly empty row block
    ("float16", 2, 7, 1, 64, 130, 45, 64),       # rep 7, ragged chunk ends
    ("bfloat16", 1, 4, 4, 128, 0, 65, 64),       # self chunk only: the first rows see one tile
    ("float16", 1, 4, 1, 64, 1340, 8, 20),       # 68 chunks: the table scan takes a second batch of 64
])
@pytest.mark.parametrize("n_split", [2, 3, 32])
def test_split_matches_closed_form(dev, dtype, B, H, H_kv, D, T_prior, T_q, chunk, n_split):
    from halo_amd.decode import ChunkRef
    rng = np.random.default_rng(17)
    T = T_prior + T_q
    q, k, v = (round_to(rng.standard_normal(s, dtype=np.float32), dtype)
               for s in ((B, H, T_q, D), (B, H_kv, T, D), (B, H_kv, T, D)))
    qg, kg, vg = (torch.from_numpy(a).to(dev).to(DT[dtype]) for a in (q, k, v))
    chunks = [ChunkRef(kg[:, :, s:min(s + chunk, T_prior)], vg[:, :, s:min(s + chunk, T_prior)], s, False)
              for s in range(0, T_prior, chunk)] + [ChunkRef(kg[:, :, T_prior:], vg[:, :, T_prior:], T_prior, True)]
    out, lse = _split(qg, chunks, n_split, q_start=T_prior)
    want, wl = A.prefill_f64(q, k, v, scale=1 / math.sqrt(D), q_start=T_prior)
    # the probabilities are rounded to the 16-bit type in front of the second product
    assert np.abs(out - want).max() <= (2e-2 if dtype == "bfloat16" else 3e-3)
    assert np.abs(lse - wl).max() <= 1e-5 * max(1.0, np.abs(wl).max())


@pytest.mark.parametrize("n_split", [1, 4])
def test_split_rows_without_keys(dev, n_split):
    """Rows in front of every causal key, and a chunk of another batch row:
    output 0 and LSE -inf where nothing is visible, alike for every split."""
    from halo_amd.decode import ChunkRef
    g = torch.Generator(device=dev).manual_seed(2)
    q = torch.randn((2, 2, 70, 64), generator=g, device=dev).to(torch.float16)
    k = torch.randn((2, 100, 64), generator=g, device=dev).to(torch.float16)
    out, lse = _split(q, [ChunkRef(k, k, 40, True, batch=1)], n_split, q_start=0)
    assert (out[0] == 0).all() and np.isneginf(lse[0]).all()
    assert (out[1, :, :40] == 0).all() and np.isneginf(lse[1, :, :40]).all()
    want, wl = A.prefill_f64(q[1:, :, 40:].float().cpu().numpy(), k[None, :, :30].float().cpu().numpy(),
                             k[None, :, :30].float().cpu().numpy(), scale=1 / 8, q_start=0)
    assert np.abs(out[1:, :, 40:] - want).max() <= 3e-3
    assert np.abs(lse[1:, :, 40:] - wl).max() <= 1e-4


def test_split_choice():
    """One pass where the query rows fill the GPU, and no more passes than
    64-row tiles or than the limit."""
    from halo_amd import _native as nat
    L = nat.lib()
    assert L.halo_prefill_splits(1, 32, 8, 4096, 128, 32768, 4096) == 1
    assert L.halo_prefill_splits(1, 32, 8, 512, 128, 60, 60) == 1
    for T_q in (1, 8, 137, 512, 1024):
        for keys in (64, 700, 9000, 10 ** 6):
            s = L.halo_prefill_splits(1, 32, 8, T_q, 128, keys, min(keys, T_q))
            assert 1 <= s <= min(32, -(-keys // 64))
            assert (L.halo_prefill_workspace_size(1, 32, 8, T_q, 128, s) > 0) == (s > 1)
