"""Page metadata and page selection at the edges of their launch rules: page
lengths on both sides of the whole-page-per-thread form, page counts off the
wave and workgroup tiles, slice counts that are no power of two, unaligned
outputs and queries, many query rows, and eligible lists out of order."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import scoring as S
from oracle.inputs import round_to

pytestmark = pytest.mark.gpu

_NAME = {torch.float32: "float32", torch.bfloat16: "bfloat16", torch.float16: "float16"}


def _rows(rng, shape, dtype):
    return round_to(rng.standard_normal(shape).astype(np.float32), _NAME[dtype])


def _t(x, dev, dtype):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev).to(dtype)


def _off(x):
    """The same values one element past a 16-byte boundary."""
    buf = torch.empty(x.numel() + 1, device=x.device, dtype=x.dtype)
    y = buf[1:].view(x.shape)
    y.copy_(x)
    return y


@pytest.mark.parametrize("dtype,D,page,P", [
    (torch.bfloat16, 128, 1, 5), (torch.bfloat16, 128, 13, 67), (torch.bfloat16, 128, 16, 129),
    (torch.bfloat16, 128, 17, 31), (torch.float16, 64, 32, 600), (torch.float16, 64, 33, 9),
    (torch.float16, 128, 11, 50),
    (torch.float32, 128, 8, 41), (torch.float32, 128, 16, 33), (torch.bfloat16, 80, 16, 19),
    (torch.float16, 256, 9, 3),
    (torch.bfloat16, 128, 145, 3), (torch.bfloat16, 128, 531, 2), (torch.float16, 64, 1100, 2),  # batches and their rest
    (torch.float32, 128, 300, 2),
])
def test_page_metadata_forms(dev, dtype, D, page, P):
    """Means and bounds are the oracle's bit for bit in both forms and into an
    unaligned output; NaN stays and zeros compare equal."""
    from halo_amd.chunk_scorer import chunk_means
    from halo_amd.quest_scorer import page_minmax
    rng = np.random.default_rng(page * 1000 + D)
    K = _rows(rng, (2, 2, P * page + page // 2, D), dtype)
    K[0, 1, 0, 3] = np.nan
    K[1, 0, :page, 5] = 0.0
    K[1, 0, :page:2, 5] = -0.0
    K[1, 1, :page, 7] = np.inf
    kt = _t(K, dev, dtype)
    kmin, kmax = page_minmax(kt, page)
    omin, omax = S.page_minmax(K, page)
    assert np.array_equal(kmin.float().cpu().numpy(), omin, equal_nan=True)
    assert np.array_equal(kmax.float().cpu().numpy(), omax, equal_nan=True)
    shape = (2, 2, P, D)
    umin, umax = _off(torch.zeros(shape, device=dev, dtype=dtype)), _off(torch.zeros(shape, device=dev, dtype=dtype))
    page_minmax(kt, page, kmin=umin, kmax=umax)
    bits = {2: torch.int16, 4: torch.int32}[kt.element_size()]
    assert torch.equal(umin.contiguous().view(bits), kmin.view(bits))
    assert torch.equal(umax.contiguous().view(bits), kmax.view(bits))
    km = chunk_means(kt, page)
    um = chunk_means(kt, page, out=_off(torch.zeros(shape, device=dev, dtype=dtype)))
    assert torch.equal(um.contiguous().view(bits), km.view(bits))
    # the row-group order: rows t = g, g + RG, ... of the page, then the groups
    RG = 256 // (D // (4 if dtype == torch.float32 else 8))
    x = K[:, :, :P * page].reshape(2, 2, P, page, D).astype(np.float32)
    total = np.zeros((2, 2, P, D), np.float32)
    for g in range(min(RG, page)):
        part = np.zeros_like(total)
        for t in range(g, page, RG):
            part = part + x[:, :, :, t]
        total = total + part
    inv = np.float32(1.0) / np.float32(page)
    if dtype == torch.float16:  # v_fma_mixlo_f16: the product is rounded once, to fp16
        total = (total.astype(np.float64) * inv).astype(np.float16).astype(np.float32)
    else:
        total = total * inv
    want = np.where(np.isfinite(total), round_to(total, _NAME[dtype]), total)  # round_to takes finite values
    assert np.array_equal(km.float().cpu().numpy(), want, equal_nan=True)


@pytest.mark.parametrize("dtype,H,H_kv,T_q,D,P,per_row,unaligned", [
    (torch.bfloat16, 32, 8, 1, 128, 9, False, False),
    (torch.float16, 9, 3, 2, 48, 65, False, True),      # 3 slices in 4 lanes
    (torch.bfloat16, 4, 4, 3, 16, 130, True, False),    # 1 slice: a page a lane
    (torch.float32, 8, 2, 5, 256, 33, False, False),    # 16 slices, 16 waves
    (torch.bfloat16, 10, 2, 40, 96, 129, False, True),  # rows split over workgroups, 6 slices
    (torch.float32, 4, 2, 33, 64, 200, True, False),
])
def test_quest_scores_forms(dev, dtype, H, H_kv, T_q, D, P, per_row, unaligned):
    from halo_amd.quest_scorer import quest_score_topk
    rng = np.random.default_rng(P)
    B = 2
    a, b = _rows(rng, (B, H_kv, P, D), dtype), _rows(rng, (B, H_kv, P, D), dtype)
    omin, omax = np.minimum(a, b), np.maximum(a, b)
    omin[0, 0, 4, 1] = np.nan
    q = _rows(rng, (B, H, T_q, D), dtype)
    qt = _t(q, dev, dtype)
    k = min(P, 40)
    idx, dots, scores = quest_score_topk(_off(qt) if unaligned else qt, _t(omin, dev, dtype), _t(omax, dev, dtype), k,
                                         per_row=per_row, want_dots=True, want_scores=True)
    assert np.array_equal(dots.cpu().numpy(), S.quest_scores(q, omin, omax, _NAME[dtype]), equal_nan=True)
    for s, r in enumerate([np.s_[i:i + 1] for i in range(B)] if per_row else [np.s_[:]]):
        ps = S.quest_page_scores(q[r], omin[r], omax[r], _NAME[dtype])
        assert np.array_equal(scores[s].cpu().numpy(), ps)
        assert idx[s].cpu().tolist() == sorted(range(P), key=lambda p: (-float(ps[p]), p))[:k]


@pytest.mark.parametrize("n,k,D,H_kv,normalize", [
    (1, 1, 128, 8, False), (64, 64, 128, 8, False), (65, 7, 48, 2, False), (257, 0, 128, 2, False),
    (512, 128, 128, 8, True), (1000, 333, 64, 4, True), (1024, 1, 256, 1, False),
])
def test_score_topk_forms(dev, n, k, D, H_kv, normalize):
    """One workgroup and the pages' own grid, and the selection of ascending and
    of shuffled lists, agree with each other: ties by lower chunk index, NaN last."""
    from halo_amd.chunk_scorer import score_topk
    rng = np.random.default_rng(n)
    dtype = torch.bfloat16
    km = _rows(rng, (1, H_kv, n, D), dtype)
    if n > 20:
        km[:, :, 11] = km[:, :, 17]
        km[:, :, 5] = np.nan
        km[:, :, 2] = 0.0
    q = _rows(rng, (1, 2 * H_kv, D), dtype)
    args = dict(normalize=normalize, beta=0.25, gamma=0.5, sink_pages=2, P_total=n)
    qt, kt = _t(q, dev, dtype), _t(km, dev, dtype)
    up = torch.arange(n, device=dev, dtype=torch.int32)
    perm = torch.from_numpy(rng.permutation(n).astype(np.int32)).to(dev)
    i0, s0 = score_topk(qt, kt, up, k, **args)
    i1, s1 = score_topk(_off(qt), kt, perm, k, **args)
    assert torch.equal(s0[0][perm.long()], s1[0])
    assert torch.equal(i0, i1)
    s = s0[0].cpu().numpy()
    want = sorted(sorted(range(n), key=lambda p: (-float(s[p]), p))[:k])
    assert i0[0].cpu().tolist() == want
    # page by page: below the size at which the scores get their own grid
    if not normalize:
        one = torch.cat([score_topk(qt, kt, up[i:i + 16].contiguous(), 1)[1][0] for i in range(0, n, 16)])
        assert torch.equal(one, s0[0])
