"""The split walk of the chunked prefill: n_split partial passes and their
merge against the float64 closed form, at the edges of the split ranges."""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import attention as A
from oracle.inputs import round_to

gpu = pytest.mark.gpu

DT = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}


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
    nb = L.halo_prefill_workspace_size(nat.dtype_code(q.dtype), B, H, H_kv, T_q, D, n_split)
    ws = torch.full((max(nb, 16),), 0xFF, device=q.device, dtype=torch.uint8)
    nat.check(L.halo_prefill_attn_split(
        q.data_ptr(), *q.stride()[:3], nat.dtype_code(q.dtype), B, H, H_kv, T_q, D, qs.data_ptr(), dd.data_ptr(),
        len(chunks), 1 / math.sqrt(D), out.data_ptr(), *out.stride()[:3], nat.dtype_code(out.dtype), lse.data_ptr(),
        n_split, ws.data_ptr(), nb, nat.stream_ptr()), "halo_prefill_attn_split")
    torch.cuda.synchronize()
    return out.cpu().numpy(), lse.cpu().numpy()


@gpu
@pytest.mark.parametrize("dtype,B,H,H_kv,D,T_prior,T_q,chunk", [
    ("bfloat16", 1, 8, 2, 128, 384, 130, 128),   # a second, nearly empty row block
    ("float16", 2, 7, 1, 64, 130, 45, 64),       # rep 7, ragged chunk ends
    ("bfloat16", 1, 4, 4, 128, 0, 65, 64),       # self chunk only: the first rows see one tile
    ("float16", 1, 4, 1, 64, 1340, 8, 20),       # 68 chunks: the table scan takes a second batch of 64
    ("float32", 1, 8, 2, 128, 384, 33, 128),     # 132 rows: a workgroup with one live wave
    ("float32", 2, 7, 1, 64, 130, 45, 64),
    ("float32", 1, 4, 1, 64, 1340, 8, 20),
])
@pytest.mark.parametrize("n_split", [1, 2, 3, 32])
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
    # (2^-9 and 2^-12 relative, of outputs below 4); fp32: sums of at most 1400 products of 2^-24
    assert np.abs(out - want).max() <= {"bfloat16": 2e-2, "float16": 3e-3, "float32": 1e-5}[dtype]
    assert np.abs(lse - wl).max() <= 1e-5 * max(1.0, np.abs(wl).max())


@gpu
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


@gpu
@pytest.mark.parametrize("T_q,prior,D", [(1, 0, 64), (31, 1, 128), (40, 65, 64), (200, 300, 64)])
@pytest.mark.parametrize("scale", [0.3, 0.0, -0.2])
def test_fp32_call(dev, T_q, prior, D, scale):
    """The public fp32 call: strided q, a head group that is no power of two,
    values behind the diagonal that are not finite, any sign of the scale."""
    from halo_amd.decode import ChunkRef
    from halo_amd.prefill import _f32_direct, prefill_attention
    rng = np.random.default_rng(T_q)
    H, H_kv, T = 6, 2, prior + T_q
    q, k, v = (rng.standard_normal(s, dtype=np.float32) for s in ((1, T_q, H, D), (1, H_kv, T, D), (1, H_kv, T, D)))
    qt = torch.from_numpy(q).to(dev).transpose(1, 2)
    kt, vt = torch.from_numpy(k).to(dev), torch.from_numpy(v).to(dev)
    chunks = [ChunkRef(kt[:, :, :prior], vt[:, :, :prior], 0, False)] if prior else []
    chunks.append(ChunkRef(kt[:, :, prior:], vt[:, :, prior:], prior, True))
    assert _f32_direct(qt, chunks)
    out, lse = prefill_attention(qt, chunks, scale=scale, return_lse=True)
    want, wl = A.prefill_f64(q.transpose(0, 2, 1, 3), k, v, scale=scale, q_start=prior)
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-5
    assert np.abs(lse.cpu().numpy() - wl).max() <= 1e-5 * max(1.0, np.abs(wl).max())
    vt[:, 0, T - 1, 3], vt[:, 1, T - 1, 5], kt[:, 0, T - 1, 0] = float("inf"), float("nan"), float("nan")
    out2 = prefill_attention(qt, chunks, scale=scale)
    assert torch.equal(out2[:, :, :-1], out[:, :, :-1])  # only the last row sees the last key
    assert out2[:, :3, -1, 3].isnan().all() and out2[:, 3:, -1, 5].isnan().all()
    assert torch.equal(out2[:, 3:, -1, :5], out[:, 3:, -1, :5])


@gpu
def test_fp32_zero_scale_of_large_scores(dev):
    """A zero scale weighs every visible key alike, however large the scores:
    of up to 1e38 here, 3e-7 relative in a weight at the fp32 maximum."""
    from halo_amd.decode import ChunkRef
    from halo_amd.prefill import prefill_attention
    rng = np.random.default_rng(8)
    q, k, v = (rng.standard_normal(s, dtype=np.float32) for s in ((1, 4, 40, 64), (1, 2, 140, 64), (1, 2, 140, 64)))
    k *= np.float32(2e36)
    qt, kt, vt = (torch.from_numpy(a).to(dev) for a in (q, k, v))
    chunks = [ChunkRef(kt[:, :, :100], vt[:, :, :100], 0, False), ChunkRef(kt[:, :, 100:], vt[:, :, 100:], 100, True)]
    out, lse = prefill_attention(qt, chunks, scale=0.0, return_lse=True)
    want, wl = A.prefill_f64(q, k, v, scale=0.0, q_start=100)
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-5
    assert np.abs(lse.cpu().numpy() - wl).max() <= 1e-5


def test_fp32_route():
    """Chunks that the matrix kernel does not read stay on the row-by-row form."""
    from halo_amd.decode import ChunkRef
    from halo_amd.prefill import _f32_direct

    class Q:  # a device query of this shape
        is_cuda, shape = True, (1, 4, 8, 64)
    k = torch.zeros((1, 2, 32, 64))
    assert _f32_direct(Q, [ChunkRef(k, k, 0, True)])
    for odd in (k[0], k.double(), torch.zeros((1, 2, 32, 66))[..., :64], k[:, :, :1].expand(1, 2, 32, 64),
                torch.zeros((2, 2, 32, 64)), torch.zeros(4098)[2:].view(1, 1, 64, 64)):
        assert not _f32_direct(Q, [ChunkRef(odd, odd, 0, True)])
    assert not _f32_direct(Q, [ChunkRef(k[0], k[0], 0, True, batch=0)])


@gpu
def test_split_choice():
    """One pass where the query rows fill the GPU, and no more passes than
    64-row tiles or than the limit."""
    from halo_amd import _native as nat
    L = nat.lib()
    assert L.halo_prefill_splits(nat.BF16, 1, 32, 8, 4096, 128, 32768, 4096) == 1
    assert L.halo_prefill_splits(nat.BF16, 1, 32, 8, 512, 128, 60, 60) == 1
    for T_q in (1, 8, 137, 512, 1024):
        for keys in (64, 700, 9000, 10 ** 6):
            s = L.halo_prefill_splits(nat.BF16, 1, 32, 8, T_q, 128, keys, min(keys, T_q))
            assert 1 <= s <= min(32, -(-keys // 64))
            assert (L.halo_prefill_workspace_size(nat.BF16, 1, 32, 8, T_q, 128, s) > 0) == (s > 1)
