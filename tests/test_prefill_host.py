"""Host side of the prefill call, without a GPU: the library is a stand-in that
records its arguments, and torch's operators are watched while the call runs."""
from __future__ import annotations

import contextlib

import numpy as np
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode


class _Lib:
    """The prefill entry points of the library."""

    def __init__(self, n_split=1, ws_bytes=0):
        self.n_split, self.ws_bytes = n_split, ws_bytes

    def halo_prefill_splits(self, *a):
        self.splits_args = a
        return self.n_split

    def halo_prefill_workspace_size(self, *a):
        return self.ws_bytes if a[-1] > 1 else 0

    def halo_prefill_attn_split(self, *a):
        self.attn_args = a
        return 0


@pytest.fixture
def host(monkeypatch):
    """prefill_attention on CPU tensors over a _Lib."""
    from halo_amd import prefill as P
    from halo_amd.decode import DESC_DTYPE
    lib = _Lib()
    monkeypatch.setattr(P.nat, "lib", lambda: lib)
    monkeypatch.setattr(P.nat, "stream_ptr", lambda s=None: 0)
    monkeypatch.setattr(P, "pack_descs", lambda chunks, **kw: (np.zeros(len(chunks), DESC_DTYPE), []))
    monkeypatch.setattr(P, "_f32_direct", lambda q, chunks: True)
    return lib


def _chunk(dtype, T=32, *, B=1, H_kv=2, D=64, **kw):
    from halo_amd.decode import ChunkRef
    shape = (H_kv, T, D) if kw.get("batch", -1) >= 0 else (B, H_kv, T, D)
    t = torch.zeros(shape, dtype=dtype)
    return ChunkRef(t, t, kw.pop("start", 0), kw.pop("causal", True), **kw)


class _Writes(TorchDispatchMode):
    """Names of the operators that allocate or write while ``inside`` is not set."""

    def __init__(self, state):
        super().__init__()
        self.state, self.outside = state, []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        name = func.overloadpacket.__name__
        if name in ("clone", "copy_", "_to_copy", "fill_") or "empty" in name:
            if not self.state["inside"]:
                self.outside.append(name)
        return out


@pytest.mark.parametrize("dtype,direct", [(torch.bfloat16, True), (torch.float32, True), (torch.float32, False)])
@pytest.mark.parametrize("q_form", ["aligned", "offset", "strided"])
def test_device_work_is_on_the_given_stream(host, monkeypatch, dtype, direct, q_form):
    """Copies of q, the output and the workspace belong to ``stream``: made
    elsewhere they would not be ordered with the kernels, and their memory
    could be handed out again while the kernels still use it."""
    from halo_amd import decode
    from halo_amd import prefill as P
    state = {"inside": False}

    @contextlib.contextmanager
    def on(stream):
        state["inside"] = True
        yield
        state["inside"] = False

    monkeypatch.setattr(torch.cuda, "stream", on)
    monkeypatch.setattr(P, "_f32_direct", lambda q, chunks: direct)
    monkeypatch.setattr(decode, "build_plan", lambda **kw: None)
    monkeypatch.setattr(decode, "launch", lambda *a, **kw: None)
    q = torch.zeros((1, 4, 8, 64), dtype=dtype)
    if q_form == "offset":
        q = torch.zeros(q.numel() + 1, dtype=dtype)[1:].view(q.shape)
    elif q_form == "strided":
        q = torch.zeros((1, 4, 8, 128), dtype=dtype)[..., ::2]
    with _Writes(state) as seen:
        P.prefill_attention(q, [_chunk(dtype)], return_lse=True, stream=object())
    assert seen.outside == []
