"""The scratch of large page selections: raw scores are kept between two
launches in a workspace and not in the caller's score buffer, which two
selections that overlap may share."""
from __future__ import annotations

import pytest
import torch


class _Lib:
    def halo_chunk_score_topk_ws(self, *a):
        self.score_out, self.workspace = a[19], a[-2]
        return 0


@pytest.mark.parametrize("given", [False, True])
def test_score_buffer_of_the_caller_is_not_scratch(monkeypatch, given):
    from halo_amd import chunk_scorer as S
    lib = _Lib()
    monkeypatch.setattr(S.nat, "lib", lambda: lib)
    monkeypatch.setattr(S.nat, "stream_ptr", lambda s=None: 0)
    q, km = torch.zeros((1, 8, 128)), torch.zeros((1, 8, 512, 128))
    elig, scores = torch.arange(512, dtype=torch.int32), torch.zeros((1, 512))
    _, out = S.score_topk(q, km, elig, 4, score_out=scores if given else None)
    assert lib.score_out == out.data_ptr() and (out is scores) == given
    assert lib.workspace and (lib.workspace != lib.score_out or not given)
    with pytest.raises(AssertionError, match="workspace"):
        S.score_topk(q, km, elig, 4, workspace=torch.zeros(511))
    S.score_topk(q, km, elig, 4, score_out=scores, workspace=scores)
    assert lib.workspace == lib.score_out == scores.data_ptr()


@pytest.mark.gpu
@pytest.mark.parametrize("n,normalize", [(64, True), (512, True), (1000, False)])
def test_one_launch_and_two_agree(dev, n, normalize):
    """halo_chunk_score_topk, without scratch, against halo_chunk_score_topk_ws
    with a workspace apart from the scores, in place of them and none."""
    from halo_amd import _native as nat
    L = nat.lib()
    g = torch.Generator(device=dev).manual_seed(n)
    q = torch.randn((1, 32, 128), generator=g, device=dev).to(torch.bfloat16)
    km = torch.randn((1, 8, n, 128), generator=g, device=dev).to(torch.bfloat16)
    elig = torch.arange(n, device=dev, dtype=torch.int32)
    k = n // 4

    def call(two, ws):
        idx = torch.full((1, k), -7, device=dev, dtype=torch.int32)
        scores = torch.full((1, n), float("nan"), device=dev)
        ws = scores if ws == "scores" else torch.full((1, n), 1e9, device=dev) if ws else None
        args = (q.data_ptr(), q.stride(0), q.stride(1), nat.BF16, 1, 32, 8, 128, km.data_ptr(), *km.stride()[:3],
                elig.data_ptr(), 0, None, n, k, 0, idx.data_ptr(), scores.data_ptr(), None, 0, None, 0, 0,
                int(normalize), 1.0, 0.5, 0.25, 64, 1, n)
        tail = (None, None, 0, None, nat.ptr(ws)) if two else ()
        fn = L.halo_chunk_score_topk_ws if two else L.halo_chunk_score_topk
        nat.check(fn(*args, *tail, nat.stream_ptr()), "score")
        torch.cuda.synchronize()
        return idx, scores

    i0, s0 = call(False, None)
    for ws in (True, "scores", None):
        i1, s1 = call(True, ws)
        assert torch.equal(i0, i1) and torch.equal(s0, s1)
